"""The matrix states of state_scan in chunks on the matrix cores and a decode step's in one kernel, against double
precision and beside the walk token by token; called as the engine calls it, with a step view."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Scan:
    def __init__(self, rule, heads, key_heads, kd, vd, lengths, seed=0, slow=True, skips=None):
        gen = torch.Generator(device=DEV).manual_seed(seed + kd + vd)
        randn = lambda *s: torch.randn(*s, generator=gen, device=DEV)
        T = sum(lengths)
        self.rule, self.H, self.G, self.kd, self.vd, self.lengths = rule, heads, key_heads, kd, vd, lengths
        self.skips = rule == 0 if skips is None else skips          # outputs take a share of the value
        self.stride = 2 * key_heads * kd + heads * vd + 4
        self.qkv, self.raw = randn(T, self.stride), randn(T, 2 * heads + 3)
        self.state = randn(len(lengths), heads, kd, vd)
        self.A_log, self.bias, self.skip = 0.5 * randn(heads), (-2.0 if slow else 1.0) + randn(heads), randn(heads)

    def run(self, chunked=True):
        """(outputs, states after) by the library."""
        from picolm_amd import kernels
        from picolm_amd.engine import program as P
        from picolm_amd.parts.calls import StateScanArgs
        P.declare(kernels.lib())
        H, G, kd, vd, T, n = self.H, self.G, self.kd, self.vd, len(self.qkv), len(self.lengths)
        order = torch.randperm(n + 1, generator=torch.Generator().manual_seed(1))[:n].int()
        state = torch.full((n + 1, 8 + H * kd * vd), 3.0, device=DEV)
        state[order.long().to(DEV), 8:] = self.state.reshape(n, -1)
        qkv, aw, out = self.qkv.clone(), torch.empty(T, 2 * H, device=DEV), torch.full((T, H * vd), 9.0, device=DEV)
        scratch = torch.full((T, H * (68 + (kd + vd if self.rule else 0))), float("nan"), device=DEV)
        args = StateScanArgs(self.rule, H, G, kd, vd, self.raw.shape[1], 3, 3 + H, self.stride, 0, G * kd, 2 * G * kd, self.A_log.data_ptr(),
                             self.bias.data_ptr(), self.skip.data_ptr() if self.skips else None, self.rule, 1e-6, kd ** -0.5, 8)
        v = P.StepView()
        v.struct_bytes, v.dtype, v.rows, v.n_tokens, v.n_seq = ctypes.sizeof(P.StepView), 0, T, T, n
        v.is_decode = int(max(self.lengths) == 1)
        cu = torch.tensor([0] + self.lengths).cumsum(0).int().to(DEV)
        new, slots = (ctypes.c_int32 * n)(*self.lengths), order.to(DEV)
        v.n_new, v.cu_seqlens, v.seq_slot = ctypes.cast(new, ctypes.POINTER(ctypes.c_int32)), cu.data_ptr(), slots.data_ptr()
        v.inp, v.out, v.in_row_bytes, v.out_row_bytes = self.raw.data_ptr(), out.data_ptr(), self.raw.shape[1] * 4, H * vd * 4
        for i, t in enumerate((qkv, aw, scratch) if chunked else (qkv, aw)):
            v.extra[i], v.extra_row_bytes[i] = t.data_ptr(), t.shape[1] * 4
        v.state, v.state_bytes_per_slot, v.n_slots = state.data_ptr(), state.shape[1] * 4, n + 1
        v.stream = torch.cuda.current_stream().cuda_stream
        f = kernels.lib().picolm_call_state_scan
        f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_void_p], ctypes.c_int
        assert f(ctypes.byref(args), ctypes.byref(v)) == 0, kernels.lib().picolm_last_error()
        torch.cuda.synchronize()
        assert bool((state[:, :8] == 3.0).all())
        return out, state[order.long().to(DEV), 8:].reshape(n, H, kd, vd)

    def reference(self):
        H, G, kd, vd = self.H, self.G, self.kd, self.vd
        d = self.qkv.double()
        q, k, v = (d[:, :G * kd].view(-1, G, kd), d[:, G * kd:2 * G * kd].view(-1, G, kd), d[:, 2 * G * kd:2 * G * kd + H * vd].view(-1, H, vd))
        if self.rule:
            q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        q, k = (x.repeat_interleave(H // G, 1) for x in (q * kd ** -0.5, k))
        soft = lambda x: torch.nn.functional.softplus(x, threshold=60.0)
        ra, rw, bias = self.raw[:, 3:3 + H].double(), self.raw[:, 3 + H:3 + 2 * H].double(), self.bias.double()
        a = torch.exp(-torch.exp(self.A_log.double()) * soft(ra + bias))
        w = torch.sigmoid(rw) if self.rule else soft(rw + bias)
        outs, states, t = [], [], 0
        for i, n in enumerate(self.lengths):
            S = self.state[i].double()
            for _ in range(n):
                S = a[t, :, None, None] * S
                u = w[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1) if self.rule else v[t])
                S = S + k[t, :, :, None] * u[:, None, :]
                outs.append((S * q[t, :, :, None]).sum(1) + (self.skip.double()[:, None] * v[t] if self.skips else 0.0))
                t += 1
            states.append(S)
        return torch.stack(outs).reshape(-1, H * vd), torch.stack(states)


def distances(got, want):
    return [float((g - w).norm() / w.norm()) for g, w in zip(got, want)]


SIZES = [(1, 4, 2, 128, 128), (1, 3, 3, 64, 48), (0, 8, 2, 128, 64), (0, 2, 1, 64, 16)]


# a chunk and a token more and less, blocks of 16, several sequences of unequal length, one of them a single token
@pytest.mark.parametrize("rule,H,G,kd,vd", SIZES)
@pytest.mark.parametrize("lengths", [[16], [33], [64], [65, 1, 17], [200, 63, 128], [16, 48], [47, 257]])
@pytest.mark.parametrize("slow", [True, False])
def test_states_in_chunks(rule, H, G, kd, vd, lengths, slow):
    x = Scan(rule, H, G, kd, vd, lengths, slow=slow)
    want = x.reference()
    got, walked = distances(x.run(), want), distances(x.run(chunked=False), want)
    print(rule, kd, vd, lengths, slow, got, "walked", walked)
    # sums of up to 200 floats, a few roundings of 2^-24 (6e-8) each; no further off than the walk but for one such
    assert max(got) < 1e-6 and all(g < 1.25 * w + 6e-8 for g, w in zip(got, walked))


@pytest.mark.parametrize("rule,H,G,kd,vd", [(1, 4, 2, 128, 128), (1, 3, 3, 64, 32), (0, 8, 2, 128, 64), (0, 2, 1, 64, 96)])
def test_a_decode_steps_states(rule, H, G, kd, vd):
    x = Scan(rule, H, G, kd, vd, [1] * 5)
    assert max(distances(x.run(), x.reference())) < 1e-6


def test_decays_of_nought_and_strong_ones_in_chunks():
    """A state that a token forgets altogether stays forgotten, and decays of 1e-30 divide nothing."""
    for rule in (0, 1):
        x = Scan(rule, 4, 2, 128, 64, [130])
        x.raw[20, 3:7], x.raw[70:90, 3:7], x.A_log[1] = 200.0, 30.0, 3.0
        assert max(distances(x.run(), x.reference())) < 2e-6


# a token in the middle of a block of 16, a block's last, a chunk's first and its last but one, the sequence's last
@pytest.mark.parametrize("rule,H,G,kd,vd", SIZES)
@pytest.mark.parametrize("at", [37, 47, 64, 126, 136])
def test_what_is_no_number_reaches_no_token_before_it(rule, H, G, kd, vd, at):
    """Queries, keys, values, strengths and decays: outputs before the token are those of a sequence without it, to the bit, and
    no number where the walk has none."""
    inf, nan = float("inf"), float("nan")
    x = Scan(rule, H, G, kd, vd, [137])
    clean = x.run()[0]
    for column, value in ((5, nan), (G * kd + 3, inf), (G * kd + kd - 1, nan), (2 * G * kd + 7, inf), (2 * G * kd + vd + 1, -inf), (("raw", 3), nan),
                          (("raw", 3 + H), nan)):
        y = Scan(rule, H, G, kd, vd, [137])
        if isinstance(column, tuple):
            y.raw[at, column[1]] = value
        else:
            y.qkv[at, column] = value
        (got, state), (walked, walked_state) = y.run(), y.run(chunked=False)
        assert torch.equal(got[:at], clean[:at]), (column, value)
        assert torch.equal(got.isfinite(), walked.isfinite()) and torch.equal(state.isfinite(), walked_state.isfinite()), (column, value)
        assert not got[at].isfinite().all()


# a prompt in chunks, one that is walked, a decode step
@pytest.mark.parametrize("lengths", [[70, 16], [15], [1, 1, 1]])
@pytest.mark.parametrize("rule,skips", [(1, True), (0, False)])
def test_either_rule_with_and_without_a_share_of_the_value(rule, skips, lengths):
    x = Scan(rule, 4, 2, 128, 64, lengths, skips=skips)
    assert max(distances(x.run(), x.reference())) < 1e-6
