"""Norms of rows whose first entries a thread keeps in registers: rows shorter than a wave, rows that fit and rows that do
not, few and many of them, against double precision; called as the engine calls them, with a step view."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def call(name, args, rows, inp, out, extras=()):
    from picolm_amd import kernels
    from picolm_amd.engine import program as P
    P.declare(kernels.lib())
    v = P.StepView()
    v.struct_bytes, v.dtype, v.rows, v.n_tokens, v.n_seq = ctypes.sizeof(P.StepView), 0, rows, rows, rows
    row_bytes = lambda t: t.shape[1] * t.element_size()
    v.inp, v.out, v.in_row_bytes, v.out_row_bytes = inp.data_ptr(), out.data_ptr(), row_bytes(inp), row_bytes(out)
    for i, t in enumerate(extras):
        if t is not None:
            v.extra[i], v.extra_row_bytes[i] = t.data_ptr(), row_bytes(t)
    v.stream = torch.cuda.current_stream().cuda_stream
    f = getattr(kernels.lib(), name)
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_void_p], ctypes.c_int
    assert f(ctypes.byref(args), ctypes.byref(v)) == 0, kernels.lib().picolm_last_error()
    torch.cuda.synchronize()


# a sum of n squares in any order is right to a few times sqrt(n) 2^-24, at most 2^-16 here; the rest are single roundings
def close(got, want):
    assert float((got.double() - want).norm() / want.norm()) <= 2e-6


def normed(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


CASES = [(1, 1), (5, 63), (1, 2048), (1030, 300), (3, 8200), (1030, 2500), (2, 10000)]


@pytest.mark.parametrize("rows,W", CASES)
def test_row_norms(rows, W):
    from picolm_amd.parts.calls import BranchNormArgs, GatedNormArgs, GatedPostnormArgs, NormedSumArgs
    gen = torch.Generator(device=DEV).manual_seed(W)
    randn = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    x, u, g, w, w2, b = randn(rows, W), randn(rows, W), randn(rows, W), randn(W), randn(W), randn(W)
    xd, ud, gd, wd, w2d, bd = (t.double() for t in (x, u, g, w, w2, b))

    got, h = x.clone(), torch.empty_like(x)
    call("picolm_call_branch_norm", BranchNormArgs(b.data_ptr(), w.data_ptr(), w2.data_ptr(), W, 1e-5, 1e-3, 0.5, 0), rows, u, got, (h,))
    want = xd + 0.5 * normed(ud + bd, wd, 1e-5)
    close(got, want)
    close(h, normed(want, w2d, 1e-3))

    got, plain = x.clone(), torch.empty_like(x)
    call("picolm_call_gated_postnorm", GatedPostnormArgs(w.data_ptr(), b.data_ptr(), W, 1.5, 1e-5), rows, u, got, (g, plain))
    want = normed(1.5 * xd + ud * torch.sigmoid(gd + bd), wd, 1e-5)
    close(got, want)
    assert torch.equal(got, plain)

    for second in (False, True):
        got = x.clone()
        args = NormedSumArgs(w.data_ptr(), w2.data_ptr() if second else None, W, 1e-5, 0.5)
        call("picolm_call_normed_sum", args, rows, u, got, (g if second else None,))
        close(got, xd + 0.5 * (normed(ud, wd, 1e-5) + (normed(gd, w2d, 1e-5) if second else 0.0)))

    for gate_first in (0, 1):
        got = torch.empty_like(x)
        call("picolm_call_gated_norm", GatedNormArgs(w.data_ptr(), W, W, W, 1e-5, gate_first, W, 0, 0, 0, 0, 0.0), rows, u, got, (g,))
        act = torch.nn.functional.silu(gd)
        close(got, normed(ud * act, wd, 1e-5) if gate_first else normed(ud, wd, 1e-5) * act)


@pytest.mark.parametrize("H,G,d,half", [(2, 1, 64, 1), (6, 3, 96, 0), (48, 4, 128, 1)])
def test_a_norm_over_all_heads_then_the_rotation(H, G, d, half):
    """Through the attention of a sequence's first token, whose output is its value, and the query rows left in the
    scratch buffer."""
    from picolm_amd.parts.calls import SinkAttentionArgs
    from picolm_amd import kernels
    from picolm_amd.engine import program as P
    P.declare(kernels.lib())
    gen = torch.Generator(device=DEV).manual_seed(H)
    randn = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    n = 3
    stride = (H + 2 * G) * d
    rows, qn, kn = randn(n, stride), randn(H * d), randn(G * d)
    cos, sin = randn(8, d // 2), randn(8, d // 2)
    q, out = torch.empty(n, H * d, device=DEV), torch.empty(n, H * d, device=DEV)
    k_pages, v_pages = torch.zeros(n, G, 64, d, device=DEV), torch.zeros(n, G, d, 64, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    pos, slots, pages, table = i32([5, 0, 7]), i32([0, 1, 2]), i32([2, 0, 1]), i32([[2], [0], [1]])
    entries = [[n, 0, 0, 0, 0, 0, 0, 0]] + [[i, 0, p, i, pg, -1, -1, -1] for i, (p, pg) in enumerate(zip([5, 0, 7], [2, 0, 1]))]
    a = SinkAttentionArgs(n_heads=H, n_kv_heads=G, head_dim=d, v_head_dim=d, in_stride=stride, q_off=0, k_off=H * d, v_off=(H + G) * d,
                          gate_off=-1, scale=1.0, eps=1e-5, q_norm=qn.data_ptr(), k_norm=kn.data_ptr(), cos_table=cos.data_ptr(),
                          sin_table=sin.data_ptr(), table_positions=8, rot_dims=d, rot_half=half, norm_all=1)
    v = P.StepView()
    work = i32(entries)
    v.struct_bytes, v.dtype, v.rows, v.n_tokens, v.n_seq, v.is_decode = ctypes.sizeof(P.StepView), 0, n, n, n, 1
    v.inp, v.out, v.in_row_bytes, v.out_row_bytes = rows.data_ptr(), out.data_ptr(), stride * 4, H * d * 4
    v.extra[0], v.extra_row_bytes[0] = q.data_ptr(), H * d * 4
    v.k_pages, v.v_pages, v.page_table, v.n_pages, v.max_pages, v.ring_pages = k_pages.data_ptr(), v_pages.data_ptr(), table.data_ptr(), n, 1, 1
    v.n_kv_heads, v.head_dim, v.v_head_dim, v.kv_writes, v.write_pages = G, d, d, 1, pages.data_ptr()
    v.tok_pos, v.seq_pos0, v.seq_slot, v.chunk_list = pos.data_ptr(), pos.data_ptr(), slots.data_ptr(), work.data_ptr()
    v.n_chunks, v.pages_per_chunk, v.most_chunks = n, 4, 1
    v.stream = torch.cuda.current_stream().cuda_stream
    f = kernels.lib().picolm_call_sink_attention
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_void_p], ctypes.c_int
    assert f(ctypes.byref(a), ctypes.byref(v)) == 0, kernels.lib().picolm_last_error()
    torch.cuda.synchronize()

    def turned(x, heads, w):
        y = normed(x.double(), w.double(), 1e-5).view(n, heads, d)
        cs, sn = (t.double()[pos.long()][:, None, :] for t in (cos, sin))
        first, second = (y[..., :d // 2], y[..., d // 2:]) if half else (y[..., 0::2], y[..., 1::2])
        a, b = first * cs - second * sn, second * cs + first * sn
        return torch.cat((a, b), -1) if half else torch.stack((a, b), -1).flatten(-2)
    close(q.view(n, H, d), turned(rows[:, :H * d], H, qn))
    key = turned(rows[:, H * d:(H + G) * d], G, kn)
    for i, (p, pg) in enumerate(zip([5, 0, 7], [2, 0, 1])):
        close(k_pages[pg, :, p, :], key[i])
        assert torch.equal(v_pages[pg, :, :, p], rows[i, (H + G) * d:].view(G, d))


def squares_in_order(x, threads):
    """Sums of the rows' squares [rows] as a workgroup of `threads` makes them in 32 bits: a thread's entries one after another
    through an FMA, a wave's threads by halves, quarters, ..., the waves one after another."""
    import numpy as np
    rows, W = x.shape
    padded = np.zeros((rows, -(-W // threads) * threads), np.float32)
    padded[:, :W] = x
    s = np.zeros((rows, threads), np.float32)
    for part in np.split(padded, padded.shape[1] // threads, 1):
        wide = part.astype(np.longdouble)                 # (a square and a sum of this size lie in 64 bits as they are)
        s = (wide * wide + s).astype(np.float32)
    s = s.reshape(rows, threads // 64, 64)
    while s.shape[2] > 1:
        s = s[:, :, :s.shape[2] // 2] + s[:, :, s.shape[2] // 2:]
    total = np.zeros(rows, np.float32)
    for w in range(threads // 64):
        total = total + s[:, w, 0]
    return total


# what is kept in registers between the passes changes no bit (rows that fit, and rows that do not)
@pytest.mark.parametrize("W", [2048, 3000, 9000])
def test_row_norms_to_the_bit(W):
    import numpy as np
    from picolm_amd.parts.calls import GatedNormArgs, GatedPostnormArgs, NormedSumArgs
    rows = 48
    gen = torch.Generator(device=DEV).manual_seed(W)
    x, u, w = (torch.randn(*s, generator=gen, device=DEV) for s in ((rows, W), (rows, W), (W,)))
    xs, us, ws = (t.cpu().numpy() for t in (x, u, w))
    fma = lambda a, b, c: (np.asarray(a, np.longdouble) * b + c).astype(np.float32)
    f32 = np.float32

    def normed_rows(rows_):
        mean = squares_in_order(rows_, 1024) / f32(W)
        return rows_ * (f32(1) / np.sqrt(mean + f32(1e-5)))[:, None] * ws
    got = torch.empty_like(x)
    call("picolm_call_gated_norm", GatedNormArgs(w.data_ptr(), W, W, W, 1e-5, 0, W, 0, 0, 0, 0, 0.0), rows, u, got)
    assert np.array_equal(got.cpu().numpy(), normed_rows(us))
    got = x.clone()
    call("picolm_call_normed_sum", NormedSumArgs(w.data_ptr(), None, W, 1e-5, 0.5), rows, u, got)
    assert np.array_equal(got.cpu().numpy(), fma(f32(0.5), normed_rows(us), xs))
    got = x.clone()
    call("picolm_call_gated_postnorm", GatedPostnormArgs(w.data_ptr(), None, W, 1.5, 1e-5), rows, u, got)
    assert np.array_equal(got.cpu().numpy(), normed_rows(fma(f32(1.5), xs, us)))
