"""Which kernel the library's rules choose for the expert products, for tests that name the kernels they are about."""

from __future__ import annotations

from research_amd import _ffi

GATE_UP, DOWN, DATA_GRADIENT, DATA_GRADIENT_PAIR = range(4)
MI355X_CUS = 256


def chosen(product, rows, reduction, columns, experts, cus=0):
    """Name of the bf16 kernel (experts = 0: a dense product; cus = 0: on the current device)."""
    return _ffi.load_library().jtmoe_product_kernel(product, rows, reduction, columns, experts, cus).decode()


def forward_kernels(rows, hidden, inter, experts=0, cus=0):
    return chosen(GATE_UP, rows, hidden, inter, experts, cus), chosen(DOWN, rows, inter, hidden, experts, cus)


def gradient_kernels(rows, hidden, inter, experts=0, cus=0):
    """Those of dZ = dY Wd^T and of dX = dG Wg^T + dU Wu^T."""
    return (chosen(DATA_GRADIENT, rows, hidden, inter, experts, cus),
            chosen(DATA_GRADIENT_PAIR, rows, inter, hidden, experts, cus))


def f32_backward_kernel(rows, hidden, inter, experts, cus=0):
    """Whether the single-precision gradients of the routed experts run in one launch ("joint") or in three."""
    return _ffi.load_library().jtmoe_f32_backward_kernel(rows, hidden, inter, experts, cus).decode()


def joint_kernels(tokens, top_k, hidden, inter, shared, experts, cus=0):
    """Those of gate/up, down, dZ and dX of routed and shared experts in one launch ("separate": in two)."""
    joint = _ffi.load_library().jtmoe_joint_kernel
    return [joint(product, tokens, top_k, hidden, inter, shared, experts, cus).decode()
            for product in (GATE_UP, DOWN, DATA_GRADIENT, DATA_GRADIENT_PAIR)]


def tiles(product, rows, reduction, columns, experts=0, cus=MI355X_CUS):
    """Name of the tiles that a bf16 product is launched in (experts = 0: a dense product)."""
    return _ffi.load_library().jtmoe_product_tiles(product, rows, reduction, columns, experts, cus).decode()


def product_tiles(rows, hidden, inter, experts=0, cus=MI355X_CUS):
    """Those of gate/up, down, dZ and dX."""
    return [tiles(GATE_UP, rows, hidden, inter, experts, cus), tiles(DOWN, rows, inter, hidden, experts, cus),
            tiles(DATA_GRADIENT, rows, hidden, inter, experts, cus), tiles(DATA_GRADIENT_PAIR, rows, inter, hidden, experts, cus)]


def joint_tiles(tokens, top_k, hidden, inter, shared, experts, cus=MI355X_CUS):
    """Those of the joint launches of routed and shared experts ("separate": in two)."""
    joint = _ffi.load_library().jtmoe_joint_tiles
    return [joint(product, tokens, top_k, hidden, inter, shared, experts, cus).decode()
            for product in (GATE_UP, DOWN, DATA_GRADIENT, DATA_GRADIENT_PAIR)]


def shared_beside(tokens, top_k, hidden, inter, shared, experts, cus=MI355X_CUS):
    """Beside which launch the shared gate/up and down products run, and in which tiles ("": neither router nor dispatch)."""
    beside = _ffi.load_library().jtmoe_shared_beside
    return [beside(product, tokens, top_k, hidden, inter, shared, experts, cus).decode() for product in (GATE_UP, DOWN)]
