"""Inputs whose edge rows decide the result, for tests of decode attention: rows at the edges of blocks, tiles and workgroup ranges get
one key that every query head of the group points along and values of their own, so that losing or misplacing one shows."""
import math

import torch


def edge_positions(n, spans):
    """First and last rows of a sequence of n rows and of its pieces of each length in spans: the first piece, one in the middle, the last."""
    at = {0, n - 1}
    for s in spans:
        for b in (s, s * (n // s // 2), s * ((n - 1) // s)):
            at |= {b - 1, b}
    return sorted(p for p in at if 0 <= p < n)


def plant(k, v, q, at, kappa=1.0):
    """k, v (n_kv, n, d) are changed in place at rows `at`; q (n_q, d) are the queries.  Together the planted rows get about half of the
    weight of an average head, whatever n is; kappa: the share of a key's projection that quantising it keeps."""
    n_kv, n, d = k.shape
    along = q.float().view(n_kv, -1, d).sum(1)                             # q_h . along is d and some noise
    score = math.log(max(n * math.exp(0.5) / len(at), math.e))             # the other scores are N(0, 1)
    k[:, at] = (along * (score * math.sqrt(d) / (d * kappa)))[:, None].to(k.dtype)
    v[:, at] *= 3


def check(got, want, q, k, v, scale, at, bound):
    """|got - want| <= bound(w, terms) elementwise, and the loss of any planted row would be more than twice that in half of the heads.

    q (n_q, d), k and v (n_kv, n, d) as the kernels see them; bound takes the weights (n_kv, n_rep, n) and the largest sum of the
    magnitudes of a score's terms (n_kv, n_rep, 1) and gives (n_kv, n_rep, d)."""
    n_kv, n, d = k.shape
    q, kt = q.float().view(n_kv, -1, d), k.float().transpose(1, 2).contiguous()
    w = torch.softmax(torch.matmul(q, kt) * scale, -1)
    b = bound(w, torch.matmul(q.abs(), kt.abs()).amax(-1, keepdim=True) * scale)
    got, want = got.float().view(b.shape), want.float().view(b.shape)
    assert ((got - want).abs() <= b).all(), float(((got - want).abs() / b).max())
    if n == 1:
        return
    for p in at:
        wp = w[:, :, p, None]
        lost = wp / (1 - wp).clamp_min(1e-6) * (v[:, None, p].float() - want).abs()
        seen = (lost > 2 * b).any(-1)
        assert seen.float().mean() >= 0.5, (p, float(seen.float().mean()))


def fp16_weights_bound(v, bits):
    """What a pass over packed keys and values may lose whose weights enter the products as fp16.

    A weight times its row's norm is rounded once (2^-11), below fp16's normal range to 2^-25 of the row's largest; the
    centroids are fp16 numbers under a scale that leaves the worst of them within 2^-13.2 at four bits and 2^-15.6 below: every element
    of a value is off by that share of the row's norm at most, and every score by that share of its terms, which moves a weight twice, in the
    numerator and in the sum."""
    eps = 2.0 ** (-13 if bits == 4 else -15)
    v = v.float()
    norm = v.norm(dim=-1, keepdim=True)

    def bound(w, terms):
        share = torch.matmul(w, v.abs())
        return (share * (2.0 ** -11 + 2 * eps * terms)
                + torch.matmul(w, norm) * eps
                + w.amax(-1, keepdim=True) * v.shape[1] * 2.0 ** -25 * v.abs().amax())
    return bound
