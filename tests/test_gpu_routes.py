"""GPU tests of dispatch edges: the one-workgroup routing at the edges of its
segments and limits, the activation fold beside it, weight packing with the
gate/up pairing in the kernel, units of up to 17 token tiles, and the GEMMs
launched alone after whatever ran before.  Each against the oracle, a plain
restatement or the general path."""
import ctypes
import dataclasses

import numpy as np
import pytest
import torch

import mini_mega_amd as mm
from mini_mega_amd import inputs

import moe_case as mc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# pairs around a segment (64), a round (1024) and the last size of the one-
# workgroup routing (4096), with few experts and the most
@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (63, 1, 8), (64, 1, 8), (65, 1, 1024), (1023, 1, 256),
                                   (1025, 1, 1024), (819, 5, 128), (4095, 1, 1024), (512, 8, 256),
                                   (4097, 1, 1024)])
def test_routing_around_the_one_workgroup_limits(T, K, E):
    rng = np.random.default_rng(T * 31 + E)
    idx = rng.integers(0, E, size=(T, K)).astype(np.int64)
    idx[rng.random((T, K)) < 0.3] = E // 2          # a hot expert, repeats within a wave
    bad = rng.random((T, K)) < 0.05
    idx[bad] = rng.choice([-1, E, E + 7, 1 << 40], size=int(bad.sum()))
    for cap in (0, max(1, T * K // (2 * E))):
        c = mc.normal_case(E, K, 256, 128, T, seed=3, scaled=False, idx=idx,
                           wts=np.full((T, K), 1.0 / K, np.float32))
        c = dataclasses.replace(c, cap=cap)
        r = mc.run_layer(c)
        mc.check_routing(c, r)
        mc.check_reduce(c, r)


# the fold runs beside the routing up to 524288 groups of 8 values (T = 512 at
# H = 8192), in a launch of its own above; T = 37: a partly filled workgroup
@pytest.mark.parametrize("T,H,scaled", [(37, 256, True), (512, 8192, True), (513, 8192, False)])
def test_fold_beside_the_routing(T, H, scaled):
    E, K, I = 4, 2, 128
    xb, xq, xsf = inputs.make_x(T, H, seed=T, scaled=scaled)
    (w1, s1), (w2, s2) = inputs.make_weights_normal(E, H, I, seed=6)
    idx, wts = inputs.route(T, E, K, seed=7)
    buf = mm.get_symm_buffer_for_mega_moe(None, E, T, K, H, I, mma_type="bf16xfp8")
    buf.x[:T].copy_(xb)
    buf.topk_idx[:T].copy_(torch.from_numpy(idx))
    buf.topk_weights[:T].copy_(torch.from_numpy(wts))
    y = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")
    mm.bf16_fp8_mega_moe(y, (w1, s1) if scaled else w1, (w2, s2) if scaled else w2, buf)
    torch.cuda.synchronize()
    L = buf.layout
    assert torch.equal(buf.workspace[L.xq:L.xq + T * H].view(T, H), xq)
    if scaled:
        assert torch.equal(buf.workspace[L.xq_sf:L.xq_sf + T * (H // 128)].view(T, H // 128), xsf)
    counts, offsets, perm, pair_pos = orc.route(idx, E, None)
    assert np.array_equal(buf.counts().cpu().numpy(), counts)
    assert np.array_equal(buf.pair_pos(T).cpu().numpy().ravel(), np.asarray(pair_pos).ravel())


# one tile column, a last workgroup of fewer than 4 column tiles, several pairs
# of blocks, the smallest pairing block; an unaligned and a strided source
@pytest.mark.parametrize("E,I,H", [(1, 128, 128), (3, 256, 640), (2, 768, 1152), (5, 512, 256)])
def test_paired_packing(E, I, H):
    G = mm.pairing_block(I)
    rng = np.random.default_rng(I + H)
    w1 = rng.integers(0, 127, size=(E, 2 * I, H)).astype(np.uint8)
    w2 = rng.integers(0, 127, size=(E, H, I)).astype(np.uint8)
    rows = inputs.paired_to_torch_rows(I)

    def check(a, b):
        p1, p2 = mm.transform_weights_for_mega_moe(a, b)
        for e in range(E):
            got = inputs.unpack_tiles(p1[e].view(torch.uint8).cpu().numpy().ravel(), 2 * I, H)
            assert np.array_equal(got, w1[e][rows])
            got = inputs.unpack_tiles(p2[e].view(torch.uint8).cpu().numpy().ravel(), H, I)
            assert np.array_equal(got, w2[e])

    a = torch.from_numpy(w1).cuda()
    b = torch.from_numpy(w2).cuda()
    fp8 = torch.float8_e4m3fn
    check(a.view(fp8), b.view(fp8))
    off = torch.empty(a.numel() + 3, dtype=torch.uint8, device="cuda")[3:].view(a.shape)
    off.copy_(a)
    check(off.view(fp8), b.view(fp8))
    check(a.transpose(1, 2).contiguous().transpose(1, 2).view(fp8), b.view(fp8))


def test_rows_that_do_not_pair_are_refused():
    w1 = torch.zeros((1, 2 * 384, 128), dtype=torch.uint8, device="cuda")   # 384 % 256 != 0
    w2 = torch.zeros((1, 128, 384), dtype=torch.uint8, device="cuda")
    with pytest.raises(RuntimeError):
        mm.transform_weights_for_mega_moe(w1.view(torch.float8_e4m3fn), w2.view(torch.float8_e4m3fn))


# rows around the largest one-unit size (272) and its multiples, and around the
# 256-row items: 257-272 run as one unit, 513-544 as two, the others as items
@pytest.mark.parametrize("rows", [[256, 257, 264, 272, 273], [512, 513, 544, 545, 1, 0, 271]])
@pytest.mark.parametrize("scaled", [True, False])
def test_units_of_seventeen_token_tiles(rows, scaled):
    """Against the oracle at the staged tolerances, and bit for bit against the
    one-launch form, which runs the items as they are; the fp8 MFMA path
    against its own result on 64-row windows (same sums, other units)."""
    E, K, H, I = len(rows), 1, 512, 256
    ids = np.repeat(np.arange(E), rows)
    np.random.default_rng(5).shuffle(ids)
    T = ids.size
    idx = ids.reshape(T, 1).astype(np.int64)
    wts = np.full((T, 1), 0.75, np.float32)
    c = mc.normal_case(E, K, H, I, T, seed=17, scaled=scaled, idx=idx, wts=wts)
    r = mc.run_layer(c)
    mc.check_routing(c, r)
    for e in range(E):
        if rows[e]:
            mc.check_l1(c, r, e, max_rows=None)
            mc.check_l2(c, r, e, max_rows=None)
    mc.check_reduce(c, r)
    r.buf.fuse_l1l2 = True
    one = mc.run_layer(c, buf=r.buf)
    assert np.array_equal(one.y32.view(np.uint32), r.y32.view(np.uint32))
    r.buf.fuse_l1l2 = False
    r.buf.mfma_fp8 = True
    f8 = mc.run_layer(c, buf=r.buf)
    buf = mm.get_symm_buffer_for_mega_moe(None, E, T, K, H, I, expert_window=64)
    buf.write_fp32_y = True
    buf.mfma_fp8 = True
    f8w = mc.run_layer(dataclasses.replace(c, win=64), buf=buf)
    assert np.array_equal(f8.y32.view(np.uint32), f8w.y32.view(np.uint32))


@pytest.mark.parametrize("mfma_fp8", [False, True])
def test_gemms_launched_alone_after_anything(mfma_fp8):
    """launch_l1 / launch_l2 run every unit whatever ran before: after a
    launch_compute that no combine followed (its L2 leaves the tail queue
    spent), and after themselves.  About 300 rows per expert, so that both
    GEMMs take tickets in every XCD range."""
    E, K, H, I, T = 32, 8, 6144, 2048, 1200
    c = mc.normal_case(E, K, H, I, T, seed=71)
    other_w2 = inputs.make_weights_normal(E, H, I, seed=72)[1]
    r = mc.run_layer(c)
    buf, L, s = r.buf, mm.lib(), torch.cuda.current_stream().cuda_stream
    buf.mfma_fp8 = mfma_fp8
    nitems, max_rows = int(r.status[1]), int(r.status[5])
    # a range of more than 64 units has a tail; the walk, which has none, is out
    assert max_rows > 128 and nitems * min(I // 128, H // 256) // 8 > 64
    y = torch.empty((T, H), dtype=torch.bfloat16, device="cuda")

    def args(l2=(c.w2, c.s2), **kw):
        a = buf.make_args(T, (c.w1, c.s1), l2, y_bf16=y)
        for k, v in kw.items():
            setattr(a, k, v)
        return ctypes.byref(a)

    def ffn():
        return buf.ffn(T * K).clone(), buf.ffn_sf(T * K).clone()

    def clear(off):
        buf.workspace[int(off):].zero_()

    def queues_zero():
        return not bool(buf.status()[44:62].any())

    assert L.mm_launch_full(args(other_w2), s) == 0
    want_other = buf.l2_out(T * K).clone()
    assert L.mm_launch_full(args(), s) == 0
    want_ffn, want_l2 = ffn(), buf.l2_out(T * K).clone()
    assert not torch.equal(want_l2, want_other)

    for before in (lambda: L.mm_launch_compute(args(), s),
                   lambda: L.mm_launch_full(args(skip_combine=1), s),
                   lambda: L.mm_launch_compute(args(skip_prologue=1), s)):
        assert before() == 0
        clear(buf.layout.l2)
        assert L.mm_launch_l2(args(), s) == 0
        assert torch.equal(buf.l2_out(T * K), want_l2)
        assert before() == 0
        assert L.mm_launch_l2(args(other_w2), s) == 0
        assert torch.equal(buf.l2_out(T * K), want_other)
        assert queues_zero()
    assert L.mm_launch_compute(args(), s) == 0
    for _ in range(2):
        clear(buf.layout.ffn)
        assert L.mm_launch_l1(args(), s) == 0
        assert all(torch.equal(a, b) for a, b in zip(ffn(), want_ffn))
        assert queues_zero()
    for _ in range(2):
        clear(buf.layout.l2)
        assert L.mm_launch_l2(args(), s) == 0
        assert torch.equal(buf.l2_out(T * K), want_l2)
        assert queues_zero()
    # and a compute on that routing after them
    clear(buf.layout.ffn)
    assert L.mm_launch_compute(args(skip_prologue=1), s) == 0
    assert torch.equal(buf.l2_out(T * K), want_l2)


@pytest.mark.parametrize("mfma_fp8", [False, True])
@pytest.mark.parametrize("T", [40, 200])
def test_few_tokens_in_a_large_workspace(T, mfma_fp8):
    """A launch sized by its tokens, in a workspace for many more, with tickets
    and stealers in both GEMMs (about 64 active experts: over 64 units of L1 and
    of L2 on each XCD; T rows on one expert): bit for bit the same tokens in a
    workspace made for them, whose grid is the general one."""
    E, K, H, I = 64, 8, 2560, 2048
    rng = np.random.default_rng(T)
    idx = np.stack([rng.permutation(E - 1)[:K] for _ in range(T)]).astype(np.int64)
    idx[:8, :] = np.arange(64).reshape(8, 8) % (E - 1)   # nearly all are active
    idx[:, 0] = E - 1                                    # and one holds T rows
    c = mc.normal_case(E, K, H, I, T, seed=T + 3, idx=idx,
                       wts=np.full((T, K), 1.0 / K, np.float32))
    runs = []
    for cap in (T, 8192):
        buf = mm.get_symm_buffer_for_mega_moe(None, E, cap, K, H, I)
        buf.mfma_fp8 = mfma_fp8
        r = mc.run_layer(c, buf=buf)
        assert int(r.status[5]) == T > 32
        for base in (16, 32):
            assert int(np.diff(r.status[base:base + 9]).min()) > 64
        n = T * K
        runs.append((r.y32.view(np.uint32), buf.ffn(n).cpu().numpy(), buf.ffn_sf(n).cpu().numpy(),
                     buf.l2_out(n).cpu().numpy()))
    assert all(np.array_equal(a, b) for a, b in zip(*runs))


# L1 ranges of exactly 64 units (no tail queue) and of 66 (the last 32 by ticket)
@pytest.mark.parametrize("active", [32, 33])
def test_ranges_around_the_smallest_with_a_tail(active):
    E, K, H, I, T = 40, 1, 256, 2048, 200
    idx = (np.arange(T) % active).astype(np.int64).reshape(T, 1)
    c = mc.normal_case(E, K, H, I, T, seed=active, idx=idx, wts=np.full((T, 1), 0.5, np.float32))
    r = mc.run_layer(c)
    assert int(np.diff(r.status[16:25]).max()) == 2 * active
    mc.check_routing(c, r)
    for e in range(active):
        mc.check_l1(c, r, e, max_rows=None)
    mc.check_reduce(c, r)
