"""bfloat16 attention with a sink and gates on the matrix cores: waves that join their results in LDS, and a sequence's
chunks combined by the workgroup that finishes last or by a merge kernel, against double precision."""
import ctypes
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import DEV, K, PagedCase, decode_work_list

pytestmark = pytest.mark.gpu


class Extras(ctypes.Structure):
    _fields_ = [("v_head_dim", ctypes.c_int32), ("bias", ctypes.c_void_p), ("bias_rows", ctypes.c_int32), ("sink", ctypes.c_void_p),
                ("gate", ctypes.c_void_p), ("gate_stride", ctypes.c_int32), ("mask_window", ctypes.c_int32), ("mask_chunk", ctypes.c_int32),
                ("out_float", ctypes.c_int32), ("keep_first", ctypes.c_int32), ("softcap", ctypes.c_float), ("gate_per_head", ctypes.c_int32),
                ("out_stride", ctypes.c_int32), ("out_mult", ctypes.c_float)]


def at(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else None


def expected(case, window, sink, gate):
    """[rows][H d] in double precision."""
    H, G, d, outs, row = case.H, case.G, case.d, [], 0
    for q, k, v, old in zip(case.q, case.k, case.v, case.lens_old):
        for t in range(old, len(q)):
            lo = max(0, t - window + 1) if window else 0
            o = np.empty((H, d))
            for h in range(H):
                s = k[lo:t + 1, h // (H // G)] @ q[t, h] / math.sqrt(d)
                top = max(s.max(), sink[h])
                p = np.exp(s - top)
                o[h] = p @ v[lo:t + 1, h // (H // G)] / (p.sum() + np.exp(sink[h] - top)) / (1 + np.exp(-gate[row, h]))
            outs.append(o.reshape(-1))
            row += 1
    return np.stack(outs)


# the result is rounded to bfloat16 (2^-9) and so are the probabilities, whose errors a sum averages: 2^-7 of the largest
def close(out, want):
    err = np.abs(out.double().cpu().numpy() - want).max()
    assert err <= 2.0 ** -7 * np.abs(want).max(), err


# one to 40 heads a group (two workgroups), each head size; chunks of one page, more than eight chunks, one chunk
@pytest.mark.parametrize("H,G,d", [(2, 2, 64), (6, 2, 96), (8, 1, 128), (32, 1, 64), (40, 1, 128)])
@pytest.mark.parametrize("pages_per_chunk,window", [(1, 0), (2, 150), (5, 0), (16, 0)])
def test_decode(H, G, d, pages_per_chunk, window):
    case = PagedCase(H, G, d, [0, 63, 64, 700, 129], [1] * 5, torch.bfloat16, seed=H * d, poison=False)
    b, lib = case.batch(), K().lib()
    gen = np.random.default_rng(1)
    sink, gate = gen.standard_normal(H).astype(np.float32), gen.standard_normal((5, H)).astype(np.float32)
    want = expected(case, window, sink, gate)
    chunk_list, n_chunks, most = decode_work_list(case, window, pages_per_chunk, spare=2)
    sink_d, gate_d = torch.from_numpy(sink).to(DEV), torch.from_numpy(gate).to(DEV)
    x = Extras(v_head_dim=d, sink=sink_d.data_ptr(), gate=gate_d.data_ptr(), gate_stride=H, gate_per_head=1)
    done = torch.zeros(K().attn_decode_counters(5, H, G), dtype=torch.int32, device=DEV)
    merged = None
    for counters in (None, done, done):          # twice: the counters must be left at zero
        out = torch.full_like(case.q_dev, float("nan"))
        partial = torch.full((5 * H * most * (d + 2),), float("nan"), device=DEV)
        assert lib.picolm_attn_decode_plain_mfma(
            at(case.q_dev), at(case.k_pages), at(case.v_pages), at(out), at(partial), 5, at(chunk_list), n_chunks, pages_per_chunk, most,
            at(b.seq_pos0), at(case.table), case.table.shape[1], case.table.shape[1], H, G, d, window, ctypes.c_float(1.0 / math.sqrt(d)),
            ctypes.byref(x), at(counters), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0, lib.picolm_last_error()
        close(out, want)
        # whoever combines the chunks, the merge kernel or the last workgroup: the same sums
        assert merged is None or torch.equal(out, merged)
        merged = out
    assert not done.any()


# one head a workgroup with the keys in turn (few tiles, or heads that four waves do not share), a head a wave
@pytest.mark.parametrize("H,G,d,old,new", [(4, 4, 64, [0, 70], [33, 31]), (6, 2, 96, [0, 5], [97, 64]), (8, 2, 128, [300, 0], [1, 65]),
                                           (64, 4, 64, [0, 40], [300, 250])])
def test_prefill(H, G, d, old, new):
    case = PagedCase(H, G, d, old, new, torch.bfloat16, seed=H + d, poison=False)
    b, lib = case.batch(), K().lib()
    gen = np.random.default_rng(2)
    sink, gate = gen.standard_normal(H).astype(np.float32), gen.standard_normal((sum(new), H)).astype(np.float32)
    sink_d, gate_d = torch.from_numpy(sink).to(DEV), torch.from_numpy(gate).to(DEV)
    x = Extras(v_head_dim=d, sink=sink_d.data_ptr(), gate=gate_d.data_ptr(), gate_stride=H, gate_per_head=1)
    tile_seq, tile_q0, n_tiles = b.prefill_tiles(lib.picolm_attn_plain_mfma_tile_rows())
    out = torch.full_like(case.q_dev, float("nan"))
    assert lib.picolm_attn_prefill_plain_mfma(
        at(case.q_dev), at(case.k_pages), at(case.v_pages), at(out), at(tile_seq), at(tile_q0), n_tiles, at(b.seq_slot),
        at(b.seq_pos0), at(b.seq_nnew), at(b.cu_seqlens), at(case.table), case.table.shape[1], case.table.shape[1], H, G, d, 0,
        ctypes.c_float(1.0 / math.sqrt(d)), ctypes.byref(x), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0, lib.picolm_last_error()
    close(out, expected(case, 0, sink, gate))


# ---- with everything that may be added ---------------------------------------------------------------------
class Added:
    """A PagedCase with values of a size of their own and what the layers add to plain attention."""

    def __init__(self, H, G, d, dv, old, new, window=0, keep_first=0, bias_rows=0, softcap=0.0, sink=False, gate="", wide=False, out_float=False,
                 seed=3):
        self.case = PagedCase(H, G, d, old, new, torch.bfloat16, seed=seed + H + d + dv, poison=False)
        self.H, self.G, self.d, self.dv, self.window, self.keep_first, self.softcap, self.gate_kind = H, G, d, dv, window, keep_first, softcap, gate
        gen, c, rows = np.random.default_rng(seed), self.case, sum(new)
        normal = lambda *s: gen.standard_normal(s).astype(np.float32)
        self.v = [torch.from_numpy(gen.standard_normal((t, G, dv))).bfloat16().double().numpy() for t in c.totals]
        pages = torch.zeros(c.k_pages.shape[0], G, dv, 64, dtype=torch.bfloat16)
        for i, t in enumerate(c.totals):
            for j in range((t + 63) // 64):
                m = min(64, t - 64 * j)
                pages[int(c.table_host[c.slots[i], j]), :, :, :m] = torch.from_numpy(self.v[i][64 * j:64 * j + m]).permute(1, 2, 0).bfloat16()
        _, order = K().kv_page_order(torch.bfloat16, dv)
        self.v_pages = torch.empty_like(pages).to(DEV)
        self.v_pages.view(*pages.shape[:2], -1)[..., order.reshape(-1).to(DEV)] = pages.reshape(*pages.shape[:2], -1).to(DEV)
        self.bias, self.sink = normal(H, bias_rows) if bias_rows else None, normal(H) if sink else None
        self.gate = normal(rows, H if gate == "head" else H * dv) if gate else None
        self.mult, self.stride = (0.75, H * dv + 5) if wide else (1.0, 0)
        self.out = torch.full((rows, self.stride or H * dv), float("nan"), dtype=torch.float32 if out_float else torch.bfloat16, device=DEV)
        self.kept = [torch.from_numpy(t).to(DEV) if t is not None else None for t in (self.bias, self.sink, self.gate)]
        address = lambda t: t.data_ptr() if t is not None else None
        self.extras = Extras(v_head_dim=dv, bias=address(self.kept[0]), bias_rows=bias_rows, sink=address(self.kept[1]), gate=address(self.kept[2]),
                             gate_stride=0 if self.gate is None else self.gate.shape[1], mask_window=0, out_float=int(out_float),
                             keep_first=keep_first, softcap=softcap, gate_per_head=int(gate == "head"), out_stride=self.stride, out_mult=self.mult)

    def want(self):
        outs, row, R = [], 0, self.H // self.G
        for q, k, v, old in zip(self.case.q, self.case.k, self.v, self.case.lens_old):
            for t in range(old, len(q)):
                seen = np.array([p for p in range(t + 1) if not self.window or p > t - self.window or p < self.keep_first])
                o = np.empty((self.H, self.dv))
                for h in range(self.H):
                    s = k[seen, h // R] @ q[t, h] / math.sqrt(self.d)
                    if self.softcap:
                        s = self.softcap * np.tanh(s / self.softcap)
                    if self.bias is not None:
                        s = s + self.bias[h, np.minimum(t - seen, self.bias.shape[1] - 1)]
                    top = s.max() if self.sink is None else max(s.max(), self.sink[h])
                    p = np.exp(s - top)
                    o[h] = p @ v[seen, h // R] / (p.sum() + (0.0 if self.sink is None else np.exp(self.sink[h] - top)))
                    if self.gate is not None:
                        g = self.gate[row, h] if self.gate_kind == "head" else self.gate[row, h * self.dv:(h + 1) * self.dv]
                        o[h] = o[h] / (1 + np.exp(-g))
                outs.append(self.mult * o.reshape(-1))
                row += 1
        return np.stack(outs)

    def work_list(self, pages_per_chunk):
        """(the list, entries, most chunks of a sequence): pages kept from the start are counted ahead of the window's."""
        from plan_reference import with_header
        entries, most = [], 1
        for i, pos in enumerate(self.case.lens_old):
            first = max(0, pos - self.window + 1) // 64 if self.window else 0
            kept = min((self.keep_first + 63) // 64, first)
            pages = list(range(kept)) + list(range(first, pos // 64 + 1))
            chunks = [pages[c:c + pages_per_chunk] for c in range(0, len(pages), pages_per_chunk)]
            most = max(most, len(chunks))
            for n, chunk in enumerate(chunks):
                phys = [int(self.case.table_host[self.case.slots[i], p]) for p in chunk[:4]]
                entries.append([i, n, pos, int(self.case.slots[i])] + phys + [-1] * (4 - len(phys)))
        return torch.from_numpy(with_header(np.array(entries, np.int32), len(entries))).to(DEV), len(entries), most

    def close(self):
        out = self.out[:, :self.H * self.dv]
        assert bool(self.out[:, self.H * self.dv:].isnan().all())
        close(out, self.want())
        return out.clone()


ADDED = [dict(bias_rows=64, sink=True, gate="entry"), dict(softcap=20.0, sink=True, gate="head", window=150, keep_first=70),
         dict(window=200, keep_first=3, wide=True, out_float=True), dict(bias_rows=7, window=100, wide=True), dict(softcap=5.0, gate="entry", out_float=True)]


# chunks of one page, of as many as come with an entry, of more, and one chunk; values narrower and wider than keys
@pytest.mark.parametrize("H,G,d,dv", [(8, 2, 128, 64), (6, 2, 64, 128), (40, 1, 96, 96)])
@pytest.mark.parametrize("pages_per_chunk", [1, 4, 6, 16])
@pytest.mark.parametrize("added", range(len(ADDED)))
def test_decode_with_everything_added(H, G, d, dv, pages_per_chunk, added):
    x = Added(H, G, d, dv, [0, 63, 70, 700, 450], [1] * 5, **ADDED[added])
    b, lib, merged = x.case.batch(), K().lib(), None
    chunk_list, n_chunks, most = x.work_list(pages_per_chunk)
    done = torch.zeros(K().attn_decode_counters(5, H, G), dtype=torch.int32, device=DEV)
    for counters in (None, done, done):
        x.out.fill_(float("nan"))
        partial = torch.full((5 * H * most * (dv + 2),), float("nan"), device=DEV)
        assert lib.picolm_attn_decode_plain_mfma(
            at(x.case.q_dev), at(x.case.k_pages), at(x.v_pages), at(x.out), at(partial), 5, at(chunk_list), n_chunks, pages_per_chunk, most,
            at(b.seq_pos0), at(x.case.table), x.case.table.shape[1], x.case.table.shape[1], H, G, d, x.window, ctypes.c_float(1.0 / math.sqrt(d)),
            ctypes.byref(x.extras), at(counters), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0, lib.picolm_last_error()
        out = x.close()
        assert merged is None or torch.equal(out, merged)
        merged = out
    assert not done.any()


# a head a wave (enough tiles of heads that four waves share), and the keys in turn
@pytest.mark.parametrize("H,G,d,dv,old,new", [(64, 4, 64, 128, [0, 40], [300, 250]), (6, 2, 128, 64, [0, 200], [97, 64]), (8, 2, 96, 96, [130], [40])])
@pytest.mark.parametrize("added", range(len(ADDED)))
def test_prefill_with_everything_added(H, G, d, dv, old, new, added):
    x = Added(H, G, d, dv, old, new, **ADDED[added])
    b, lib = x.case.batch(), K().lib()
    tile_seq, tile_q0, n_tiles = b.prefill_tiles(lib.picolm_attn_plain_mfma_tile_rows())
    assert lib.picolm_attn_prefill_plain_mfma(
        at(x.case.q_dev), at(x.case.k_pages), at(x.v_pages), at(x.out), at(tile_seq), at(tile_q0), n_tiles, at(b.seq_slot),
        at(b.seq_pos0), at(b.seq_nnew), at(b.cu_seqlens), at(x.case.table), x.case.table.shape[1], x.case.table.shape[1], H, G, d, x.window,
        ctypes.c_float(1.0 / math.sqrt(d)), ctypes.byref(x.extras), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0, lib.picolm_last_error()
    x.close()
