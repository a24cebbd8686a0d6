"""The picked experts of a few rows (a decode batch), whose weights are streamed once for all pairs, against double
precision; called as the engine calls it, with a step view."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Experts:
    def __init__(self, E, D, F, identity=0, act=0, weight_on_input=0, seed=0):
        gen = torch.Generator(device=DEV).manual_seed(seed + E * 1000 + D + F)
        randn = lambda *s: torch.randn(*s, generator=gen, device=DEV)
        self.E, self.D, self.F, self.identity, self.act, self.on_input, self.gen = E, D, F, identity, act, weight_on_input, gen
        self.gate, self.up = ((randn(E, F, D) / D ** 0.5).bfloat16() for _ in range(2))
        self.down = (randn(E, D, F) / F ** 0.5).bfloat16()

    def picks(self, rows, top):
        """[rows, 2 top] words: the picks, every row's own ones differing, and their weights."""
        ids = torch.stack([torch.randperm(self.E + self.identity, generator=self.gen, device=DEV)[:top] for _ in range(rows)]).int()
        w = torch.rand(rows, top, generator=self.gen, device=DEV) + 0.1
        return ids, w, torch.cat([ids, w.view(torch.int32)], 1).contiguous()

    def run(self, h, words, top, out, adds, streamed=True, pair_rows=None):
        from picolm_amd import kernels
        from picolm_amd.engine import program as P
        from picolm_amd.parts.calls import RoutedExpertsArgs
        rows = len(h)
        P.declare(kernels.lib())
        act, y = torch.full((rows, top * self.F), 7.0, device=DEV), torch.full((rows, top * self.D if pair_rows is None else pair_rows), 7.0, device=DEV)
        plan = torch.zeros(rows, top + self.E + 1, device=DEV)
        args = RoutedExpertsArgs(self.gate.data_ptr(), self.up.data_ptr(), self.down.data_ptr(), 1, self.E, top, self.D, self.F, int(adds),
                                 self.identity, self.act, 7.0, 1.702, self.on_input)
        v = P.StepView()
        v.struct_bytes, v.dtype, v.rows, v.n_tokens = ctypes.sizeof(P.StepView), 1, rows, rows
        v.inp, v.out, v.in_row_bytes, v.out_row_bytes = h.data_ptr(), out.data_ptr(), self.D * 2, self.D * 4
        for i, t in enumerate((words, act, y, plan) if streamed else (words, act)):
            v.extra[i], v.extra_row_bytes[i] = t.data_ptr(), t.shape[1] * 4
        v.stream = torch.cuda.current_stream().cuda_stream
        f = kernels.lib().picolm_call_routed_experts
        f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_void_p], ctypes.c_int
        assert f(ctypes.byref(args), ctypes.byref(v)) == 0, kernels.lib().picolm_last_error()
        torch.cuda.synchronize()
        return out

    def reference(self, h, ids, w, out, adds):
        h, total = h.double(), out.double() if adds else torch.zeros_like(out, dtype=torch.float64)
        for k in range(ids.shape[1]):
            for e in range(self.E):
                rows = (ids[:, k] == e).nonzero()[:, 0]
                x, wk = h[rows], w[rows, k, None].double()
                g, u = x @ self.gate[e].double().T, x @ self.up[e].double().T
                if self.on_input:
                    g, u = g * wk, u * wk
                if self.act:
                    g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
                    unit = g * torch.sigmoid(1.702 * g) * (u + 1.0)
                else:
                    unit = g * torch.sigmoid(g) * u
                total[rows] += (1.0 if self.on_input else wk) * (unit @ self.down[e].double().T)
            same = (ids[:, k] >= self.E).nonzero()[:, 0]
            total[same] += w[same, k, None].double() * h[same]
        return total


def check(x, rows, top, adds=False, seed=0):
    h = torch.randn(rows, x.D, generator=x.gen, device=DEV).bfloat16()
    ids, w, words = x.picks(rows, top)
    out = torch.randn(rows, x.D, generator=x.gen, device=DEV)
    want = x.reference(h, ids, w, out, adds)
    got = x.run(h, words, top, out.clone(), adds)
    return float((got - want).norm() / want.norm()), float((got - want).abs().max() / want.abs().max())


# up to four, eight and 16 pairs of an expert at a time and more than that, from 64 rows on tiles of 16 pairs, 16, 32 and 64 at a
# time; fewer pairs than experts; one expert; widths that are one line, no power of two, and less than the four waves' lines
@pytest.mark.parametrize("E,D,F", [(1, 64, 64), (8, 2048, 2048), (3, 192, 320), (40, 320, 192), (2, 128, 1344)])
@pytest.mark.parametrize("rows", [1, 2, 7, 16, 17, 33, 63, 64, 100, 255])
def test_streamed_experts(E, D, F, rows):
    x = Experts(E, D, F)
    top = min(E, 2 if rows % 2 else 3)
    norm, worst = check(x, rows, top, adds=rows % 2 == 1)
    # exact products, float sums of up to 2,048 of them: a few roundings of 2^-24 each, with the hidden units' own; steps of
    # 64 rows and more with many pairs an expert go through tiles that round the hidden units to eight bits (2^-9 each).  Which
    # steps keep them in 32 bits is what the library promises, and said here again: a step that no longer did would fail
    streamed = rows < 64 or rows * top <= 20 * E
    assert norm < (2e-6 if streamed else 4e-3) and worst < (1e-5 if streamed else 2e-2), (E, D, F, rows, norm, worst)


# up to four and eight pairs of an expert at a time and more of them, one expert, fewer pairs than experts; widths below 512
# columns, that end inside 512, and inside a workgroup's weight rows
@pytest.mark.parametrize("E,D,F", [(8, 2048, 2048), (1, 64, 64), (3, 200, 328), (40, 320, 192), (2, 1032, 2568)])
@pytest.mark.parametrize("rows", [1, 2, 7, 16, 33, 63])
def test_streamed_experts_are_those_of_a_workgroup_per_pair_to_the_bit(E, D, F, rows):
    """However many of its rows a step brings an expert: the same sums in the same order, so that a router behind them that is not
    sure of a pick decides as it did."""
    for x, top in ((Experts(E, D, F), min(E, 2)), (Experts(E, D, F, identity=2), 3), (Experts(E, D, F, act=1, weight_on_input=1), min(E, 3))):
        h = torch.randn(rows, D, generator=x.gen, device=DEV).bfloat16()
        ids, w, words = x.picks(rows, top)
        out = torch.randn(rows, D, generator=x.gen, device=DEV)
        for adds in (True, False):
            assert torch.equal(x.run(h, words, top, out.clone(), adds), x.run(h, words, top, out.clone(), adds, streamed=False))


def test_streamed_experts_of_more_pairs_than_a_workgroup_lists_at_a_time():
    x = Experts(40, 64, 64)
    h = torch.randn(63, 64, generator=x.gen, device=DEV).bfloat16()
    ids, w, words = x.picks(63, 20)
    out = torch.zeros(63, 64, device=DEV)
    assert torch.equal(x.run(h, words, 20, out.clone(), False), x.run(h, words, 20, out.clone(), False, streamed=False))


@pytest.mark.parametrize("rows", [3, 40])
def test_streamed_experts_identity_picks_clamps_and_weights_on_the_input(rows):
    assert check(Experts(4, 128, 192, identity=3), rows, 5)[0] < 2e-6
    assert check(Experts(4, 128, 192, act=1, weight_on_input=1), rows, 3)[0] < 2e-6


def test_streamed_experts_of_a_row_do_not_depend_on_the_other_rows():
    x = Experts(4, 256, 192)
    h = torch.randn(40, 256, generator=x.gen, device=DEV).bfloat16()
    ids, w, words = x.picks(40, 2)
    whole = x.run(h, words, 2, torch.zeros(40, 256, device=DEV), False)
    for first, rows in ((0, 1), (5, 9), (20, 20)):
        part = x.run(h[first:first + rows].contiguous(), words[first:first + rows].contiguous(), 2, torch.zeros(rows, 256, device=DEV), False)
        assert torch.equal(part, whole[first:first + rows])


def test_streamed_experts_pass_on_what_is_no_number():
    """An infinity or a NaN in a row stays in that row, and is no number there."""
    x = Experts(2, 128, 64)
    h = torch.randn(20, 128, generator=x.gen, device=DEV).bfloat16()
    h[3, 5], h[11, 7] = float("inf"), float("nan")
    ids, w, words = x.picks(20, 2)
    got, want = x.run(h, words, 2, torch.zeros(20, 128, device=DEV), False), x.reference(h, ids, w, torch.zeros(20, 128, device=DEV), False)
    bad = torch.zeros(20, dtype=torch.bool, device=DEV)
    bad[3] = bad[11] = True
    assert torch.equal(got.isfinite().all(1), ~bad) and not got[11].isfinite().any()
    assert torch.equal(got[3].isfinite(), want[3].isfinite())
    assert float((got[~bad] - want[~bad]).abs().max()) < 1e-5


@pytest.mark.parametrize("rows", [16, 63])
def test_few_rows_do_without_room_for_the_pairs_outputs(rows):
    """A scratch buffer that is too short for the pairs' outputs is no error where the kernels of a workgroup per pair
    need none."""
    x = Experts(8, 256, 192)
    h = torch.randn(rows, 256, generator=x.gen, device=DEV).bfloat16()
    ids, w, words = x.picks(rows, 2)
    out = torch.zeros(rows, 256, device=DEV)
    assert torch.equal(x.run(h, words, 2, out.clone(), False, pair_rows=2 * 256 - 1), x.run(h, words, 2, out.clone(), False))
