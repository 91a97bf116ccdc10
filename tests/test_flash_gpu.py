"""The prompt attention kernel (bh::launch_flash_prefill, which the Qwen3 engine
runs for every prefill chunk) against 64-bit softmax attention: row counts
around the 32-vector wave and the workgroup, positions around the 32-key tile
and the KS-tile step, every group size, both head widths, both caches, slabs
and a shuffled paged pool; and its independence of how a prompt is chunked.

Tolerance: the kernel claims the precision of f32, so the bar is what f32
arithmetic of the plain formula shows on the same data: 1.25 times its error in
the 2-norm (plus 2^-24, the rounding of a result, where one key or few leave the
plain formula without an error of its own) and twice its largest error."""
import ctypes as C

import numpy as np
import pytest
import torch

from brain_amd import load

pytestmark = pytest.mark.gpu


def flash():
    fn = load().bh_flash_prefill_rows
    fn.restype, fn.argtypes = C.c_int, [C.c_void_p] * 9 + [C.c_uint32] * 9 + [C.c_float, C.c_uint32]
    return fn


class Setup:
    def __init__(self, nseq, npos, nkv, group, hd, kv8, paged, seed=0):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        self.nseq, self.nkv, self.group, self.hd, self.kv8 = nseq, nkv, group, hd, kv8
        self.nh, self.max_seq = nkv * group, npos + 3
        hkv = nkv * hd
        if paged:
            bs = 32 if npos < 300 else 96
            self.max_bt = (self.max_seq + bs - 1) // bs
            self.nblk = nseq * self.max_bt + 1
            bt = torch.randperm(self.nblk, device="cuda", generator=g)[: nseq * self.max_bt].view(nseq, -1)
            slots, self.bs = self.nblk * bs, bs
            self.bt = bt.to(torch.int32).contiguous()
            at = torch.arange(npos, device="cuda")
            self.slot = bt[:, at // bs] * bs + at % bs
        else:
            self.bt, self.bs, self.max_bt, self.nblk = None, 0, 0, 0
            slots = nseq * self.max_seq
            self.slot = torch.arange(nseq, device="cuda")[:, None] * self.max_seq + torch.arange(npos, device="cuda")
        if kv8:
            self.k, self.v = (torch.randint(-127, 128, (slots, hkv), device="cuda", generator=g, dtype=torch.int8) for _ in "kv")
            self.ks, self.vs = ((torch.rand(slots, nkv, device="cuda", generator=g) + 0.5) / 70 for _ in "kv")
        else:
            self.k, self.v = (torch.randn(slots, hkv, device="cuda", generator=g) for _ in "kv")
            self.ks = self.vs = None
        self.q = torch.randn(nseq, npos, self.nh, hd, device="cuda", generator=g)
        self.scale = hd ** -0.5

    def run(self, p0, p1):
        """Context of rows p0..p1 of every sequence."""
        n = p1 - p0
        q = self.q[:, p0:p1].clone(memory_format=torch.contiguous_format)  # the kernel writes over it
        pos = torch.arange(p0, p1, device="cuda", dtype=torch.int32).repeat(self.nseq)
        seq = torch.arange(self.nseq, device="cuda", dtype=torch.int32).repeat_interleave(n)
        ptr = lambda t: None if t is None else t.data_ptr()  # noqa: E731
        rc = flash()(torch.cuda.current_stream().cuda_stream, q.data_ptr(), ptr(self.k), ptr(self.v), ptr(self.ks),
                     ptr(self.vs), pos.data_ptr(), seq.data_ptr(), ptr(self.bt), self.nh, self.nkv, self.hd, n, self.nseq,
                     self.max_seq, self.max_bt, self.bs, self.nblk, self.scale, self.kv8)
        assert rc == 0
        torch.cuda.synchronize()
        return q

    def ref(self, p0, p1, dtype):
        out = torch.empty(self.nseq, p1 - p0, self.nh, self.hd, device="cuda", dtype=dtype)
        mask = torch.arange(p1, device="cuda")[None, :] > torch.arange(p0, p1, device="cuda")[:, None]
        for b in range(self.nseq):
            sl = self.slot[b, :p1]
            k, v = (x[sl].to(dtype).view(p1, self.nkv, self.hd) for x in (self.k, self.v))
            if self.kv8:
                k, v = k * self.ks[sl].to(dtype)[:, :, None], v * self.vs[sl].to(dtype)[:, :, None]
            for h in range(self.nh):
                s = (self.q[b, p0:p1, h].to(dtype) @ k[:, h // self.group].t()) * self.hd ** -0.5
                out[b, :, h] = torch.softmax(s.masked_fill(mask, -float("inf")), -1) @ v[:, h // self.group]
        return out


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("nseq,npos,nkv,group,hd,paged", [
    (1, 1, 1, 1, 128, False), (2, 15, 2, 2, 64, False), (1, 33, 2, 4, 128, True), (3, 64, 1, 8, 64, True),
    (1, 127, 1, 3, 128, False), (2, 129, 2, 5, 64, True), (1, 257, 1, 7, 128, True), (1, 1030, 2, 2, 128, False),
    (2, 515, 1, 6, 64, False),
])
def test_flash_prefill_matches_softmax(gpu, kv8, nseq, npos, nkv, group, hd, paged):
    s = Setup(nseq, npos, nkv, group, hd, kv8, paged, seed=npos)
    for p0, p1 in {(0, npos), (npos // 3, npos), (npos - 1, npos)}:
        got, want = s.run(p0, p1).double(), s.ref(p0, p1, torch.float64)
        plain = s.ref(p0, p1, torch.float32).double() - want
        err = float((got - want).norm() / want.norm())
        print(p0, p1, "error", err, "plain f32", float(plain.norm() / want.norm()))
        assert err < 1.25 * float(plain.norm() / want.norm()) + 2.0 ** -24
        assert (got - want).abs().max() < 2 * plain.abs().max() + 1e-6


def test_flash_prefill_keeps_the_bits_of_a_product(gpu):
    """Two keys of the same score: k0 by one product x y of significands whose
    bf16 parts leave the most out, k1 by three products of x with the bf16
    parts of y, which leave nothing out; values 1 and 0, so that the context is
    the weight of k0, 1/2. x y is off by at most 2^-24 for its parts, and each
    score by 2^-24 (k0) and twice that (k1) for its sums; a weight by 1/4 of
    the difference."""
    n, hd = 256, 128
    s = Setup(n, 2, 1, 1, hd, False, False, seed=4)
    s.scale = 1.0
    rng = np.random.default_rng(4)

    def worst(m):  # near a tie of the first part and of the second
        top = rng.integers(0, 4, m) << 16
        low = np.where(rng.random(m) < 0.5, 0xFF00 + rng.integers(0, 256, m), 0x7F00 + rng.integers(0, 512, m))
        return (0x3F800000 + top + low).astype(np.uint32).view(np.float32) * np.float32(64)

    x, y = worst(n), worst(n)
    x[0] = y[0] = np.uint32(0x3F80FFFF).view(np.float32) * np.float32(64)
    parts, rest = [], torch.from_numpy(y)
    for _ in range(3):
        parts.append(rest.to(torch.bfloat16).float())
        rest = rest - parts[-1]
    assert not rest.any()
    s.q.zero_(), s.k.zero_(), s.v.zero_()
    s.q[:, 1, 0, 7:10] = torch.from_numpy(x).cuda()[:, None]
    s.k[s.slot[:, 0], 7] = torch.from_numpy(y).cuda()
    s.k[s.slot[:, 1], 7:10] = torch.stack(parts, 1).cuda()
    s.v[s.slot[:, 0]] = 1.0
    got = s.run(0, 2)[:, 1, 0].double().cpu().numpy()
    score = x.astype(np.float64) * y
    assert (np.abs(got - 0.5) <= 0.25 * 4 * 2.0 ** -24 * score[:, None] + 2.0 ** -24).all()


@pytest.mark.parametrize("kv8", [False, True])
@pytest.mark.parametrize("hd,group,nkv", [(128, 2, 2), (64, 5, 2), (128, 2, 8), (64, 1, 16)])
def test_flash_prefill_chunking_gives_the_same_bits(gpu, kv8, hd, group, nkv):
    """With 8 and 16 kv heads the whole prompt takes the workgroups of twice the
    rows (f32 cache, above 128 of them), the chunks those of split columns."""
    s = Setup(2, 300, nkv, group, hd, kv8, True, seed=9)
    whole = s.run(0, 300)
    cuts = [0, 1, 2, 35, 64, 191, 300]
    parts = torch.cat([s.run(a, b) for a, b in zip(cuts, cuts[1:])], 1)
    assert torch.equal(whole, parts)


def plain64(s, p1):
    """Context of rows 0..p1 in numpy float64, each row over its visible keys alone."""
    q, kc, vc, slot = (t.cpu().numpy() for t in (s.q, s.k, s.v, s.slot))
    out = np.empty((s.nseq, p1, s.nh, s.hd))
    with np.errstate(all="ignore"):
        for b in range(s.nseq):
            k, v = (x[slot[b]].reshape(-1, s.nkv, s.hd).astype(np.float64) for x in (kc, vc))
            if s.kv8:
                k, v = (x * sc.cpu().numpy()[slot[b]][:, :, None].astype(np.float64) for x, sc in ((k, s.ks), (v, s.vs)))
            for i in range(p1):
                for h in range(s.nh):
                    sc = (q[b, i, h].astype(np.float64) * k[: i + 1, h // s.group]).sum(1) * s.hd ** -0.5
                    w = np.exp(sc - np.fmax.reduce(sc))
                    out[b, i, h] = (w[:, None] * v[: i + 1, h // s.group]).sum(0) / w.sum()
    return out


@pytest.mark.parametrize("hd,group", [(128, 2), (64, 3)])
@pytest.mark.parametrize("what", ["v_nan", "v_inf", "v_top", "k_low", "k_nan", "q_nan", "vs_inf", "ks_nan"])
def test_flash_prefill_values_at_the_ends_of_f32(gpu, what, hd, group):
    """A value that is not finite, or rounds to an infinity in bf16, or scores
    far below any other key, in one cache slot: rows before it do not see it
    (a masked key is left out, not weighted with zero), rows from it on are
    what the formula gives, and neither depends on the chunking. The 2-norm
    bar is the one of the finite cases."""
    kv8 = what in ("vs_inf", "ks_nan")
    s = Setup(2, 75, 2, group, hd, kv8, True, seed=21)
    at = s.slot[0, 0 if what == "k_low" else 37]
    if what == "v_nan":
        s.v[at, 5] = float("nan")
    elif what == "v_inf":
        s.v[at, 5] = float("inf")
    elif what == "v_top":
        s.v[at, 5] = torch.finfo(torch.float32).max
    elif what == "q_nan":
        s.q[0, 40, 1, 3] = float("nan")
    elif what == "k_nan":
        s.k[at, 5] = float("nan")
    elif what == "k_low":  # row 0 sees this key alone; its score is finite and below -1e34
        s.q.abs_()
        s.k[at] = -1e36
    elif what == "vs_inf":
        s.vs[at, 0] = float("inf")
        s.v[at] = torch.where(s.v[at] == 0, torch.ones_like(s.v[at]), s.v[at])  # no 0 x infinity in the formula
    else:
        s.ks[at, 0] = float("nan")
    want = plain64(s, 75)
    for cuts in ([0, 75], [0, 20, 38, 39, 64, 75]):
        got = torch.cat([s.run(a, b) for a, b in zip(cuts, cuts[1:])], 1).double().cpu().numpy()
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        fin = np.isfinite(want)
        assert np.array_equal(got[~fin & ~np.isnan(want)], want[~fin & ~np.isnan(want)])
        scale = np.where(fin, np.abs(want), 0).max((0, 1, 2))  # one column holds numbers of another size
        err = np.abs(np.where(fin, got, 0) - np.where(fin, want, 0))
        assert (err <= 1e-5 * np.maximum(scale, 1)).all()
