"""What a correct W4 head may give: the bf16 values between the roundings of ref - e and ref + e, e the
float32 error of its sums."""
from __future__ import annotations

import torch


def w4_limits(x: torch.Tensor, w: torch.Tensor, mag: torch.Tensor):
    """x [M, K], w [N, K] the dequantized weight and mag [N, K] the size of what the kernels multiply x
    with (|q + 128| + |zero + 128| times the scale), float64 -> (low, high) of the logits [M, N].

    A group's 128 products are summed twice in float32, times the code and for the offset: at most
    2 x 128 roundings, each of at most 2^-24 of a partial sum. The products have random signs, so the
    partial sums are within a few T_g = sqrt(sum over the group of (x mag)^2), and were all the roundings
    of a group to go one way, its error would be 256 2^-24 T_g. The groups' errors are independent: e =
    256 2^-24 sqrt(sum of T_g^2). (Adding the groups up is small beside it: G roundings of sums that
    the offset has left.) Rounding to bf16 is monotonic, so every value within e rounds to within
    the roundings of the two ends."""
    ref = x @ w.T
    e = 256 * 2.0 ** -24 * ((x * x) @ (mag * mag).T).sqrt()
    return (ref - e).bfloat16().double(), (ref + e).bfloat16().double()
