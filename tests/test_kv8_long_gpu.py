"""The paged scores and apply kernels at the sizes where their chunking can go
wrong: sequence lengths around the 128-position chunk and its multiples, block
sizes with and without a factor of 4, a table longer than the part staged at a
time, head_dim below, at and above the 64-wide workgroup, groups of one to
32 heads, and table entries outside the pool. Bit for bit against the
oracle, which sums in the same order."""
import numpy as np
import pytest
import torch

from brain_amd import load
from brain_amd._lib import check
from oracle import oracle as o

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("lens,bs,n_kv,group,hd", [
    ([1, 127, 128, 129], 16, 2, 2, 128),
    ([255, 256, 257, 383, 384, 385], 32, 1, 1, 64),
    ([513, 640, 3], 5, 2, 3, 36),
    ([700, 130], 6, 1, 5, 128),
    ([300, 64], 4, 1, 2, 256),
    ([2049, 2048, 6001], 1, 1, 2, 64),   # 6001 table entries: three staged parts
    ([1029, 0, 77], 16, 2, 2, 72),
    ([200, 3], 16, 2, 9, 64), ([70, 513, 1], 32, 1, 32, 128),  # sets of two heads and a rest
    ([2100] + [2000] * 31, 32, 2, 3, 64), ([1400] * 24, 32, 1, 7, 128),  # of the whole group; of four and three
])
def test_paged_scores_apply_chunk_edges(gpu, lens, bs, n_kv, group, hd):
    rng = np.random.default_rng(sum(lens) + bs)
    batch, nh = len(lens), n_kv * group
    cap = max(lens)
    max_bt = (cap + bs - 1) // bs
    nblk = batch * max_bt
    bt = rng.permutation(nblk).reshape(batch, max_bt).astype(np.uint32)
    pool = rng.integers(0, 2 ** 32, nblk * bs * n_kv * hd // 4, dtype=np.uint32)
    sc = rng.uniform(0.01, 0.05, nblk * bs * n_kv).astype(np.float32)
    q = rng.standard_normal((batch, nh, hd)).astype(np.float32)
    probs = rng.random((batch, nh, cap)).astype(np.float32)
    pre = np.full((batch, nh, cap), 7.0, np.float32)
    ln = np.array(lens, np.uint32)
    scale = float(np.float32(1.0 / np.sqrt(hd)))
    want_s = o.paged_decode_scores_i8(q, pool, bt, lens, sc, pre, nh, group, hd, bs, n_kv * hd, cap, scale)
    want_c = o.paged_decode_apply_i8(probs, pool, bt, lens, sc, nh, group, hd, bs, n_kv * hd, cap)
    lib, st = load(), torch.cuda.current_stream().cuda_stream
    d = {k: dev(v.view(np.int32) if v.dtype == np.uint32 else v)
         for k, v in dict(q=q, probs=probs, pool=pool, sc=sc, bt=bt, ln=ln, s=pre).items()}
    ctx = torch.empty(batch, nh, hd, device="cuda")
    shape = (batch, nh, group, hd, bs, n_kv * hd, cap, max_bt)

    def run(pool_words):
        check(lib.bh_paged_decode_scores_i8(st, d["q"].data_ptr(), d["pool"].data_ptr(), pool_words, d["bt"].data_ptr(),
                                            d["ln"].data_ptr(), d["sc"].data_ptr(), sc.size, d["s"].data_ptr(), *shape,
                                            scale))
        check(lib.bh_paged_decode_apply_i8(st, d["probs"].data_ptr(), d["pool"].data_ptr(), pool_words,
                                           d["bt"].data_ptr(), d["ln"].data_ptr(), d["sc"].data_ptr(), sc.size,
                                           ctx.data_ptr(), *shape))
        return d["s"].cpu().numpy(), ctx.cpu().numpy()

    got_s, got_c = run(pool.size)
    assert np.array_equal(got_s.view(np.uint32).ravel(), np.asarray(want_s, np.float32).view(np.uint32).ravel())
    assert np.array_equal(got_c.view(np.uint32).ravel(), np.asarray(want_c, np.float32).view(np.uint32).ravel())
    # Half the pool declared: the entries past it are skipped, as if their
    # probabilities were zero and their scores never written.
    words = pool.size // 2
    per_slot = n_kv * hd
    dead = np.zeros((batch, cap, n_kv), bool)
    for b in range(batch):
        j = np.arange(cap)
        slot = bt[b, j // bs].astype(np.int64) * bs + j % bs
        for h in range(n_kv):
            dead[b, :, h] = (slot * per_slot + h * hd + hd + 3) // 4 > words
    mask = np.repeat(dead.transpose(0, 2, 1), group, axis=1)
    d["s"].copy_(dev(pre))
    got_s, got_c = run(words)
    live = np.arange(cap)[None, None, :] < ln[:, None, None]
    ws = np.where(mask | ~live, pre, np.asarray(want_s, np.float32).reshape(pre.shape))
    assert np.array_equal(got_s.view(np.uint32).ravel(), ws.view(np.uint32).ravel())
    wc = o.paged_decode_apply_i8(np.where(mask, np.float32(0), probs), pool, bt, lens, sc, nh, group, hd, bs, n_kv * hd, cap)
    assert np.array_equal(got_c.ravel(), np.asarray(wc, np.float32).ravel())


@pytest.mark.parametrize("lens,bs,nh,group", [
    ([5, 200, 129], 2 ** 32 - 1, 4, 2), ([5, 200, 129], 2 ** 32 - 4, 4, 2), ([5, 200, 129], 2 ** 32 - 16, 2, 1),
    ([5, 200, 129], 256, 4, 2 ** 32 - 1), ([5, 200, 129], 256, 5, 3),
])
def test_paged_sizes_near_the_end_of_32_bits(gpu, lens, bs, nh, group):
    """One block holds every position; a sum with its size or with the group's would wrap."""
    rng = np.random.default_rng(5)
    batch, hd, n_kv, cap, slots = len(lens), 64, (nh - 1) // group + 1, max(lens), 256
    bt, ln = np.zeros((batch, 1), np.uint32), np.array(lens, np.uint32)
    pool = rng.integers(0, 2 ** 32, slots * n_kv * hd // 4, dtype=np.uint32)
    sc = rng.uniform(0.01, 0.05, slots * n_kv).astype(np.float32)
    q = rng.standard_normal((batch, nh, hd)).astype(np.float32)
    probs = rng.random((batch, nh, cap)).astype(np.float32)
    pre = np.full((batch, nh, cap), 7.0, np.float32)
    # The oracle with one block of the pool's size and a group of the heads: the same slots.
    obs, og = slots, min(group, nh)
    want_s = o.paged_decode_scores_i8(q, pool, bt, lens, sc, pre, nh, og, hd, obs, n_kv * hd, cap, 0.125)
    want_c = o.paged_decode_apply_i8(probs, pool, bt, lens, sc, nh, og, hd, obs, n_kv * hd, cap)
    lib, st = load(), torch.cuda.current_stream().cuda_stream
    d = {k: dev(v.view(np.int32) if v.dtype == np.uint32 else v)
         for k, v in dict(q=q, probs=probs, pool=pool, sc=sc, bt=bt, ln=ln, s=pre).items()}
    ctx = torch.empty(batch, nh, hd, device="cuda")
    shape = (batch, nh, group, hd, bs, n_kv * hd, cap, 1)
    check(lib.bh_paged_decode_scores_i8(st, d["q"].data_ptr(), d["pool"].data_ptr(), pool.size, d["bt"].data_ptr(),
                                        d["ln"].data_ptr(), d["sc"].data_ptr(), sc.size, d["s"].data_ptr(), *shape, 0.125))
    check(lib.bh_paged_decode_apply_i8(st, d["probs"].data_ptr(), d["pool"].data_ptr(), pool.size, d["bt"].data_ptr(),
                                       d["ln"].data_ptr(), d["sc"].data_ptr(), sc.size, ctx.data_ptr(), *shape))
    assert np.array_equal(d["s"].cpu().numpy().view(np.uint32).ravel(), np.asarray(want_s, np.float32).view(np.uint32).ravel())
    assert np.array_equal(ctx.cpu().numpy().view(np.uint32).ravel(), np.asarray(want_c, np.float32).view(np.uint32).ravel())
