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
