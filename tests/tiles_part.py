"""What the tiles of a 16-bit backward compute, apart from the label's entry.

By default the label's entry of the logits' gradient is added to the results in fp32, outside the tiles.  It is most of either
gradient: with a vocabulary of some ten thousand a whole slice of the rest can be lost without passing a hundredth of the whole, so a
test of the tiles looks at the rest alone."""

import torch

from oracle import lce_oracle as O


def check_tiles_part(dh32, dw32, g_lp, g_ent, h, w, y, tau=1.0):
    """fp32 gradients (either may be None) without the label's entry, against float64, in the relative 2-norm.  Every element of the
    logits' gradient is rounded to 8 significant bits (fp16: 11, fewer below 6e-5), by up to 2^-8 of itself; the errors are independent,
    and so are the signs of a sum's terms, so that the result is off by less than 2^-8 of its own 2-norm (0.2 to 0.4 of that on
    such inputs, where a lost tenth of the vocabulary is a fifth of the norm)."""
    want_h, want_w = O.lce_backward(g_lp, g_ent, h, w, y, tau, compute_dtype=torch.float64)
    share = (g_lp / tau).double()[:, None]
    if dh32 is not None:
        label = share * w[y].double()
        want, got = want_h.double() - label, dh32.double() - label
        assert want.norm() == 0 or ((got - want).norm() / want.norm()).item() <= 2.0**-8, ((got - want).norm() / want.norm()).item()
    if dw32 is not None:
        label = torch.zeros_like(want_w, dtype=torch.float64).index_add_(0, y, share * h.double())
        want, got = want_w.double() - label, dw32.double() - label
        assert want.norm() == 0 or ((got - want).norm() / want.norm()).item() <= 2.0**-8, ((got - want).norm() / want.norm()).item()
    return want_h, want_w
