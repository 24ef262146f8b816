"""The window-sum kernel at the edges of its chunks (256 elements of a
window, four per lane) and rows (columns around the 64 lanes of a wave),
writing and adding, against Kronecker products in numpy.

Blocking of SZ environment sectors with the fermionic site: every window is
f * (+-1) * A * b of one environment block and one site element, so an
element is a sum of at most two products: 1e-15 relative."""
import ctypes as C

import numpy as np
import pytest
import torch

from b2g import _lib as L
from b2g import dmrg, states as Q

pytestmark = pytest.mark.gpu

SITE = [(0, 0), (1, -1), (1, 1), (2, 0)]


def q(n, tw):
    return Q.q_make(Q.SZ, n, 0, tw, 0)


@pytest.mark.parametrize("dims", [
    (1, 1, 2), (1, 63, 5), (64, 4, 65), (3, 85, 256), (257, 1, 130)])
@pytest.mark.parametrize("add", [0, 1])
def test_window_edges(gpu_ctx, dims, add):
    print("dims", dims, "add", add, flush=True)
    dev = gpu_ctx.device
    secs = sorted((q(3 + i, (3 + i) % 2), d) for i, d in enumerate(dims))
    env = Q.StateInfo([s for s, _ in secs], [d for _, d in secs])
    site = Q.StateInfo(sorted(q(*s) for s in SITE), [1] * 4)
    ref = sorted({Q.q_add(Q.SZ, int(a), int(b)) for a in env.q
                  for b in site.q})
    fused = Q.tensor_product(Q.SZ, env, site,
                             Q.StateInfo(ref, [0] * len(ref)))

    def ops(basis, types):
        t = dmrg.OpTensor(Q.SZ, basis, basis, list(range(len(types))),
                          [q(*x) for x in types], dev)
        g = torch.Generator(device=dev).manual_seed(len(types))
        t.data.normal_(generator=g)
        return t

    # C0 = A0 (x) 1 + A1 (x) c, C1 = A1 (x) 1 (types (0,0) and (1,1))
    a = ops(env, [(0, 0), (1, 1)])
    b = ops(site, [(0, 0), (-1, -1)])
    c = ops(fused, [(0, 0), (1, 1)])
    if not add:  # a plan clears C up to its last window only
        c.data.zero_()
    terms = [(0, 0, 0, 1.0), (0, 1, 1, -0.5), (1, 1, 0, 2.0)]
    keep, d = [], L.b2g_contract()
    d.symmetry = Q.SZ
    d.bra_a = d.ket_a = dmrg._sinfo(env, keep)
    d.bra_b = d.ket_b = dmrg._sinfo(site, keep)
    d.bra = d.ket = dmrg._sinfo(fused, keep)
    d.n_a_infos, d.a_info_dq, d.a_infos, d.n_a_ops, d.a_ops = a.c_side(keep)
    d.n_b_infos, d.b_info_dq, d.b_infos, d.n_b_ops, d.b_ops = b.c_side(keep)
    d.n_c_infos, d.c_info_dq, d.c_infos, d.n_c_ops, d.c_ops = c.c_side(keep)
    tm = (L.b2g_contract_term * len(terms))(
        *[L.b2g_contract_term(i, x, y, 0, f) for i, x, y, f in terms])
    d.n_terms, d.terms = len(terms), tm

    want = c.data.cpu().numpy().copy() if add else np.zeros(c.data.numel())
    start, size = {}, {}
    for i, qa in enumerate(int(v) for v in env.q):
        for qb in (int(v) for v in site.q):
            s = Q.q_add(Q.SZ, qa, qb)
            start[qa, qb] = size.get(s, 0)
            size[s] = size.get(s, 0) + int(env.n[i])
    ah, bh = a.data.cpu().numpy(), b.data.cpu().numpy()
    for i, x, y, f in terms:
        la, lb, lc = a.layout(x), b.layout(y), c.layout(i)
        for ia in range(len(la)):
            ka, m, n = int(la.quanta[ia]), int(la.nbra[ia]), int(la.nket[ia])
            o = a.off[x] + int(la.shift[ia])
            A = ah[o:o + m * n].reshape(m, n)
            sign = -1.0 if lb.fermion and Q.q_n(ka) % 2 else 1.0
            for ib in range(len(lb)):
                kb = int(lb.quanta[ib])
                ic = lc.find(Q.q_add(Q.SZ, ka, kb))
                r0 = start[Q.q_add(Q.SZ, ka, la.dq),
                           Q.q_add(Q.SZ, kb, lb.dq)]
                k0 = start[ka, kb]
                ld, o = int(lc.nket[ic]), c.off[i] + int(lc.shift[ic])
                W = want[o:o + int(lc.nbra[ic]) * ld].reshape(-1, ld)
                W[r0:r0 + m, k0:k0 + n] += f * sign * A * bh[
                    b.off[y] + int(lb.shift[ib])]
    h = C.c_void_p()
    lib = L.lib()
    L.check(lib.b2g_contract_plan(gpu_ctx.h, C.byref(d), 0, C.byref(h)))
    torch.cuda.synchronize()
    L.check(lib.b2g_winplan_run(h, a.data.data_ptr(), b.data.data_ptr(),
                                c.data.data_ptr(), add))
    gpu_ctx.synchronize()
    L.check(lib.b2g_winplan_destroy(h))
    got = c.data.cpu().numpy()
    assert np.abs(got - want).max() <= 1e-15 * np.abs(want).max()
