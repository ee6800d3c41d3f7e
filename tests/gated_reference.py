"""Gated products in 64 bits, and how far from them a kernel may be whose two sums are off by so much."""

import torch


def gated(sums, off, activation="silu", limit=None):
    """act(g) * u for sums [M, 2 N] = [g, u] in float64, and the bound of a bfloat16 result's error where a sum is off by up to ``off``:
    the gates' slopes are at most 1.13; the result's rounding (eight bits: 2^-8) and the float32 arithmetic between (2^-20 of the
    halves, the exponential of an argument of up to 88 in size included)."""
    n = sums.shape[1] // 2
    g, u, off_g, off_u = sums[:, :n], sums[:, n:], off[:, :n], off[:, n:]
    if activation == "clamped":
        g, u = g.clamp(max=limit), u.clamp(-limit, limit) + 1
        act = g * torch.sigmoid(1.702 * g)
    else:
        act = torch.nn.functional.silu(g) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    want = act * u
    return want, 1.15 * off_g * (u.abs() + off_u) + act.abs() * off_u + 2.0 ** -8 * want.abs() + 2.0 ** -20 * (g * u).abs() + 1e-30


def rounded(sums):
    """What a whole number is off by once it is rounded to bfloat16: nothing up to 256."""
    return torch.where(sums.abs() <= 256, 0.0, 2.0 ** -8 * sums.abs())
