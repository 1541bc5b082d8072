"""GPU parity of chunked (segmented) prefill and of the mixed batch against
the CPU oracle (restated reference segmented path and float64 math)."""
import pytest
import torch

from oracle import decode as OD
from oracle import segmented as OSg
from vllm_neuron_amd import _kernels as K
from vllm_neuron_amd import workloads as W
from vllm_neuron_amd.functional import mixed_batch_attention, segmented_attention

from test_prefill_plan import even_bytes, workspace_bytes

pytestmark = pytest.mark.gpu

TOL_BF16 = 2e-2
TOL_FP8 = 6e-2


def _seq_kv(cache, table_row, n, H):
    return torch.stack([OD.gather_contiguous(cache, table_row, n, h) for h in range(H)])


PREFILL_CASES = [
    # q_heads, kv_heads, d, bs, new, prior, window, sink, tp_q, tp_out
    (8, 2, 128, 32, 96, 64, 0, False, True, False),
    (8, 2, 64, 16, 130, 0, 0, False, True, True),
    (12, 2, 128, 64, 200, 128, 0, True, False, False),
    (16, 2, 64, 32, 160, 96, 64, True, True, True),
    (4, 4, 128, 16, 33, 48, 0, False, True, False),
    (8, 1, 64, 32, 257, 512, 128, False, True, False),
    # head dims staged through zero-padded rows (attention_segmented_cte.py:783-790: d <= 128)
    (8, 2, 80, 32, 130, 64, 0, False, True, False),
    (12, 2, 96, 16, 200, 128, 64, True, False, True),
    (4, 4, 48, 32, 96, 32, 0, False, True, False),
]


@pytest.mark.parametrize("case", range(len(PREFILL_CASES)))
def test_segmented_vs_reference(gpu, case):
    Hq, Hkv, d, bs, S, prior, win, use_sink, tp_q, tp_out = PREFILL_CASES[case]
    cfg = W.PrefillConfig("t", 1, Hq, Hkv, d, bs, S, prior, prior, seed=50 + case)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    q = b.q.transpose(0, 1).contiguous()  # [Nh, S, D]
    if not tp_q:
        q = q.transpose(1, 2).contiguous()
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(case)).to(gpu) if use_sink else None
    scale = d ** -0.5
    out = segmented_attention(q, b.k_cache, b.v_cache, b.block_table, b.prior.view(1, 1), bs, 0,
                              scale=scale, tp_q=tp_q, tp_out=tp_out, sliding_window=win or None,
                              sink=None if sink is None else sink.view(Hq, 1))
    ref = OSg.ref_segmented_attention(q.cpu(), b.k_cache.cpu(), b.v_cache.cpu(),
                                      b.block_table.cpu(), b.prior.cpu().view(1, 1), bs, scale,
                                      tp_q=tp_q, tp_out=tp_out, sliding_window=win or None,
                                      sink=None if sink is None else sink.cpu().view(Hq, 1))
    assert out.shape == ref.shape
    err = (out.float().cpu() - ref.float()).abs().max().item()
    assert err <= TOL_BF16, err
    # float64 math on the contiguous sequence
    n = prior + S
    ks = _seq_kv(b.k_cache.cpu(), b.block_table[0].cpu(), n, Hkv)
    vs = _seq_kv(b.v_cache.cpu(), b.block_table[0].cpu(), n, Hkv)
    f = OSg.fp32_prefill(b.q.cpu(), ks, vs, prior, scale, win, None if sink is None else sink.cpu())
    o = out.float().cpu()
    o = o.transpose(1, 2) if tp_out else o
    err64 = (o.transpose(0, 1).double() - f).abs().max().item()
    assert err64 <= TOL_BF16, err64


def test_varlen_matches_per_sequence(gpu):
    """The 4 x 512 chunked-prefill sub-batch (priors U[0, 4096]) in one
    varlen launch equals one segmented_attention call per sequence."""
    cfg = W.PREFILL_CONFIGS["llama3_8b_prefill_4x512"]
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    out = K.paged_prefill(b.q, b.cu_seqlens, b.prior, b.max_seqlen_q, b.k_cache, b.v_cache,
                          b.block_table, scale=cfg.head_dim ** -0.5)
    for i in range(cfg.num_seqs):
        s0, s1 = int(b.cu_seqlens[i]), int(b.cu_seqlens[i + 1])
        q = b.q[s0:s1].transpose(0, 1).contiguous()
        ref = OSg.ref_segmented_attention(q.cpu(), b.k_cache.cpu(), b.v_cache.cpu(),
                                          b.block_table[i:i + 1].cpu(), b.prior[i:i + 1].cpu(),
                                          cfg.block_size, cfg.head_dim ** -0.5)
        err = (out[s0:s1].transpose(0, 1).float().cpu() - ref.float()).abs().max().item()
        assert err <= TOL_BF16, (i, err)


@pytest.mark.parametrize("d,packed", [(128, False), (96, False), (96, True)])
def test_fp8_prefill_per_head_scales(gpu, d, packed):
    from vllm_neuron_amd.functional.attention.attention_decode import _swizzle_packed_k
    cfg = W.PrefillConfig("t", 1, 12, 2, d, 64, 160, 128, 128, fp8=True, seed=77)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache, quant_mode=2,
               k_scale=b.k_quant, v_scale=b.v_quant, scale_per_head=True)
    q = b.q.transpose(0, 1).contiguous()
    kc_in = _swizzle_packed_k(b.k_cache) if packed else b.k_cache
    out = segmented_attention(q, kc_in, b.v_cache, b.block_table, b.prior.view(1, 1),
                              cfg.block_size, 0, fp8_packed=packed, k_dequant_scale=b.k_dequant,
                              v_dequant_scale=b.v_dequant)
    # oracle: the reference semantics once per kv head with scalar folding
    # (scale * s_k[h], output * s_v[h])
    G = cfg.q_heads // cfg.kv_heads
    for h in range(cfg.kv_heads):
        sl = slice(h * G, (h + 1) * G)
        kc = b.k_cache[:, h:h + 1].cpu().float()
        vc = b.v_cache[:, h:h + 1].cpu().float()
        ref = OSg.ref_segmented_attention(q[sl].cpu().float(), kc, vc, b.block_table.cpu(),
                                          b.prior.cpu().view(1, 1), cfg.block_size,
                                          cfg.head_dim ** -0.5 * float(b.k_dequant[h]))
        ref = ref * float(b.v_dequant[h])
        err = (out[sl].float().cpu() - ref).abs().max().item()
        assert err <= TOL_FP8, (h, err)


def test_mixed_batch_equals_composition(gpu):
    """One mixed call (4 prefill chunks + decode rows) equals the reference
    composition: segmented_attention per prefill sequence and the decode
    path for the decode rows, over the same cache."""
    pcfg = W.PrefillConfig("mp", 2, 16, 2, 128, 32, 96, 0, 300, seed=81)
    pb = W.make_prefill_batch(pcfg, gpu)
    dcfg = W.DecodeConfig("md", 3, 16, 2, 128, 32, 40, 500, seed=82)
    db = W.make_decode_batch(dcfg, gpu)
    # one cache pool: append the decode batch's blocks after the prefill's
    nb_p = pb.k_cache.shape[0]
    kc = torch.cat([pb.k_cache, db.k_cache], 0)
    vc = torch.cat([pb.v_cache, db.v_cache], 0)
    dt = torch.where(db.block_table >= 0, db.block_table + nb_p, db.block_table)
    dslots = db.slots + nb_p * dcfg.block_size
    kc_ref, vc_ref = kc.clone(), vc.clone()
    out_d, out_p = mixed_batch_attention(
        kc, vc, q_decode=db.q, k_decode=db.k_new, v_decode=db.v_new, decode_block_table=dt,
        decode_pos_ids=db.pos, decode_slots=dslots, q_prefill=pb.q, k_prefill=pb.k_new,
        v_prefill=pb.v_new, prefill_slots=pb.slots, prefill_cu_seqlens=pb.cu_seqlens,
        prefill_prior=pb.prior, prefill_block_table=pb.block_table,
        max_seqlen_q=pb.max_seqlen_q)
    # composition, step by step
    K.kv_write(pb.k_new, pb.v_new, pb.slots, kc_ref, vc_ref)
    for i in range(pcfg.num_seqs):
        s0, s1 = int(pb.cu_seqlens[i]), int(pb.cu_seqlens[i + 1])
        q = pb.q[s0:s1].transpose(0, 1).contiguous()
        ref = OSg.ref_segmented_attention(q.cpu(), kc_ref.cpu(), vc_ref.cpu(),
                                          pb.block_table[i:i + 1].cpu(), pb.prior[i:i + 1].cpu(),
                                          pcfg.block_size, pcfg.head_dim ** -0.5)
        err = (out_p[s0:s1].transpose(0, 1).float().cpu() - ref.float()).abs().max().item()
        assert err <= TOL_BF16, (i, err)
    f = OD.fp32_decode(db.q.cpu(), db.k_new.cpu(), db.v_new.cpu(), kc_ref.cpu().float(),
                       vc_ref.cpu().float(), dt.cpu(), db.pos.cpu(), scale=dcfg.head_dim ** -0.5)
    err = (out_d.float().cpu().double() - f).abs().max().item()
    assert err <= TOL_BF16, err
    # the decode rows' new K/V landed in their slots
    K.kv_write(db.k_new.reshape(-1, 2, 128), db.v_new.reshape(-1, 2, 128), dslots, kc_ref, vc_ref)
    assert torch.equal(kc.cpu(), kc_ref.cpu()) and torch.equal(vc.cpu(), vc_ref.cpu())


def test_prefill_empty_and_fully_masked(gpu):
    """prior 0, window 1 (each row sees itself only) and a sequence of 0
    rows in a varlen batch."""
    cfg = W.PrefillConfig("t", 2, 8, 2, 64, 16, 40, 0, 0, seed=91)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    cu = torch.tensor([0, 40, 40], dtype=torch.int32, device=gpu)  # second sequence empty
    out = K.paged_prefill(b.q[:40], cu, b.prior, 40, b.k_cache, b.v_cache, b.block_table,
                          scale=64 ** -0.5, sliding_window=1)
    # window 1: output row r = V[r] of its own kv head
    v = _seq_kv(b.v_cache.cpu(), b.block_table[0].cpu(), 40, 2)  # [2, 40, 64]
    ref = v.repeat_interleave(4, 0).transpose(0, 1)
    assert (out.float().cpu() - ref.float()).abs().max().item() <= 1e-2


@pytest.mark.parametrize("split", [1 << 20, 0])
def test_long_table_small_blocks(gpu, split):
    """Block size 16 and a 12288-token prior: unsplit, one key chunk spans
    772 blocks, more block offsets than the workgroup's threads stage in
    one pass; split in halves (the default), 416 and 356.  Both match
    float64 math."""
    cfg = W.PrefillConfig("long", 1, 8, 2, 128, 16, 64, 12288, 12288, seed=93)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    assert b.block_table.shape[1] * 16 >= 12288 + 64
    scale = 128 ** -0.5
    out = K.paged_prefill(b.q, b.cu_seqlens, b.prior, 64, b.k_cache, b.v_cache, b.block_table,
                          scale=scale, split_tokens=split)
    n = 12288 + 64
    ks = _seq_kv(b.k_cache.cpu(), b.block_table[0].cpu(), n, 2)
    vs = _seq_kv(b.v_cache.cpu(), b.block_table[0].cpu(), n, 2)
    f = OSg.fp32_prefill(b.q.cpu(), ks, vs, 12288, scale, 0, None)
    err = (out.float().cpu().double() - f).abs().max().item()
    assert err <= TOL_BF16, err


SPLIT_CASES = [
    # q_heads, kv_heads, d, bs, new, priors, window, sink, fp8
    (32, 8, 128, 32, 256, [1500, 96, 700], 0, False, False),   # copy-ring kernel
    (16, 2, 128, 32, 200, [900, 0], 0, True, False),
    (16, 2, 64, 32, 160, [1200, 64], 64, True, False),         # d = 64 kernel, window
    (12, 2, 128, 64, 128, [1024, 320], 0, False, True),        # fp8 cache
]


@pytest.mark.parametrize("case", range(len(SPLIT_CASES)))
@pytest.mark.parametrize("split", [64, 192, 512])
def test_split_keys_match_unsplit_and_reference(gpu, case, split):
    """Key ranges cut into chunks of `split` keys (partials merged by the
    combine kernel) give the unsplit result, and both match the reference
    per sequence; sequences of very different lengths share the launch."""
    Hq, Hkv, d, bs, S, priors, win, use_sink, fp8 = SPLIT_CASES[case]
    pmax = max(priors)  # pool and table sized for the longest sequence
    cfg = W.PrefillConfig("s", len(priors), Hq, Hkv, d, bs, S, pmax, pmax, fp8=fp8,
                          seed=90 + case)
    b = W.make_prefill_batch(cfg, gpu)
    # replace the priors (the generator draws one value for every sequence)
    pr = torch.tensor(priors, dtype=torch.int32)
    tot = pr + S
    nblk = b.block_table.shape[1]
    need = int(((tot + bs - 1) // bs).max())
    if need > nblk:
        pytest.skip("table too narrow for the chosen priors")
    kw = {}
    if fp8:
        kw = dict(k_dequant=b.k_dequant, v_dequant=b.v_dequant)
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache, quant_mode=2,
                   k_scale=b.k_quant, v_scale=b.v_quant, scale_per_head=True)
    # fresh table: every sequence gets distinct random blocks for its span
    nb = b.k_cache.shape[0]
    g = torch.Generator().manual_seed(5 + case)
    perm = torch.randperm(nb - 1, generator=g) + 1
    table = torch.full((len(priors), nblk), -1, dtype=torch.int32)
    off = 0
    for i in range(len(priors)):
        n = int((tot[i] + bs - 1) // bs)
        if off + n > nb - 1:
            pytest.skip("pool too small for the chosen priors")
        table[i, :n] = perm[off:off + n].to(torch.int32)
        off += n
    table = table.to(gpu)
    prior = pr.to(gpu)
    sink = torch.randn(Hq, generator=g).to(gpu) if use_sink else None
    scale = d ** -0.5
    base = K.paged_prefill(b.q, b.cu_seqlens, prior, S, b.k_cache, b.v_cache, table,
                           scale=scale, sliding_window=win, sink=sink,
                           split_tokens=1 << 20, **kw)
    out = K.paged_prefill(b.q, b.cu_seqlens, prior, S, b.k_cache, b.v_cache, table,
                          scale=scale, sliding_window=win, sink=sink, split_tokens=split, **kw)
    # chunks keep their own running max, so the bf16 rounding of the
    # probabilities differs: allow two bf16 ulps at |o| ~ 2
    assert (out.float() - base.float()).abs().max().item() <= 1.6e-2
    tol = TOL_FP8 if fp8 else TOL_BF16
    for i in range(len(priors)):
        s0, s1 = int(b.cu_seqlens[i]), int(b.cu_seqlens[i + 1])
        n = int(tot[i])
        kc, vc = b.k_cache.cpu(), b.v_cache.cpu()
        if fp8:
            kc = kc.float() * b.k_dequant.cpu().view(1, -1, 1, 1)
            vc = vc.float() * b.v_dequant.cpu().view(1, -1, 1, 1)
        ks = _seq_kv(kc, table[i].cpu(), n, Hkv)
        vs = _seq_kv(vc, table[i].cpu(), n, Hkv)
        f = OSg.fp32_prefill(b.q[s0:s1].cpu(), ks, vs, priors[i], scale, win,
                             None if sink is None else sink.cpu())
        err = (out[s0:s1].float().cpu().double() - f).abs().max().item()
        assert err <= tol, (i, err)


@pytest.mark.parametrize("fp8", [False, True])
def test_copy_ring_and_register_kernels_agree(gpu, fp8):
    """A d = 128 cache (bf16, or FP8 widened in the ring) runs the copy-ring
    kernel, whose copies share the block offsets of K and V; a V cache with
    its own block stride (a view of a wider allocation) takes the
    register-staged kernel.  Both match float64 math, and each other to
    within two bf16 steps."""
    priors = [700, 96]
    cfg = W.PrefillConfig("r", len(priors), 16, 4, 128, 32, 160, max(priors), max(priors),
                          fp8=fp8, seed=131)
    b = W.make_prefill_batch(cfg, gpu)
    kw = {}
    if fp8:
        kw = dict(k_dequant=b.k_dequant, v_dequant=b.v_dequant)
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache, quant_mode=2,
                   k_scale=b.k_quant, v_scale=b.v_quant, scale_per_head=True)
    else:
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    nb, Hkv, bs, d = b.v_cache.shape
    wide = torch.zeros(nb, Hkv + 1, bs, d, dtype=b.v_cache.dtype, device=gpu)
    wide[:, :Hkv].copy_(b.v_cache)
    v_view = wide[:, :Hkv]
    assert v_view.stride(0) != b.k_cache.stride(0)
    prior = torch.tensor(priors, dtype=torch.int32, device=gpu)
    scale = d ** -0.5
    ring = K.paged_prefill(b.q, b.cu_seqlens, prior, cfg.new_tokens, b.k_cache, b.v_cache,
                           b.block_table, scale=scale, **kw)
    regs = K.paged_prefill(b.q, b.cu_seqlens, prior, cfg.new_tokens, b.k_cache, v_view,
                           b.block_table, scale=scale, **kw)
    assert (ring.float() - regs.float()).abs().max().item() <= 1.6e-2
    kc, vc = b.k_cache.cpu(), b.v_cache.cpu()
    if fp8:
        kc = kc.float() * b.k_dequant.cpu().view(1, -1, 1, 1)
        vc = vc.float() * b.v_dequant.cpu().view(1, -1, 1, 1)
    for i, pr in enumerate(priors):
        s0, s1 = int(b.cu_seqlens[i]), int(b.cu_seqlens[i + 1])
        n = pr + (s1 - s0)
        ks = _seq_kv(kc, b.block_table[i].cpu(), n, Hkv)
        vs = _seq_kv(vc, b.block_table[i].cpu(), n, Hkv)
        f = OSg.fp32_prefill(b.q[s0:s1].cpu(), ks, vs, pr, scale, 0, None)
        for out in (ring, regs):
            err = (out[s0:s1].float().cpu().double() - f).abs().max().item()
            assert err <= (TOL_FP8 if fp8 else TOL_BF16), (i, err)


@pytest.mark.parametrize("fp8", [False, True])
def test_compact_kernel_matches_reference(gpu, fp8):
    """``compact_kernel`` (the launch that fits beside a decode workgroup:
    the 4-wave copy ring for bf16, the register-staged kernel for FP8) on a
    multi-sequence batch with a long prior (split keys) against float64 math
    and the default launch."""
    cfg = W.PrefillConfig("t", 3, 16, 2, 128, 32, 300, 0, 3600, fp8=fp8, seed=91)
    b = W.make_prefill_batch(cfg, gpu)
    kw = {}
    if fp8:
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache, quant_mode=2,
                   k_scale=b.k_quant, v_scale=b.v_quant, scale_per_head=True)
        kw = dict(k_dequant=b.k_dequant, v_dequant=b.v_dequant)
    else:
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    scale = cfg.head_dim ** -0.5
    run = lambda compact: K.paged_prefill(b.q, b.cu_seqlens, b.prior, b.max_seqlen_q, b.k_cache,
                                          b.v_cache, b.block_table, scale=scale,
                                          compact_kernel=compact, **kw)
    got, base = run(True).float().cpu(), run(False).float().cpu()
    tol = TOL_FP8 if fp8 else TOL_BF16
    assert (got - base).abs().max().item() <= tol / 2
    cu = b.cu_seqlens.cpu().tolist()
    kc, vc = b.k_cache.cpu().float(), b.v_cache.cpu().float()
    kd = b.k_dequant.cpu() if fp8 else torch.ones(cfg.kv_heads)
    vd = b.v_dequant.cpu() if fp8 else torch.ones(cfg.kv_heads)
    for i in range(len(cu) - 1):
        prior = int(b.prior[i])
        n = prior + cu[i + 1] - cu[i]
        row = b.block_table[i].cpu()
        ks = _seq_kv(kc, row, n, cfg.kv_heads) * kd.view(-1, 1, 1)
        vs = _seq_kv(vc, row, n, cfg.kv_heads) * vd.view(-1, 1, 1)
        f = OSg.fp32_prefill(b.q[cu[i]:cu[i + 1]].cpu(), ks, vs, prior, scale)
        err = (got[cu[i]:cu[i + 1]].double() - f).abs().max().item()
        assert err <= tol, (i, err)


@pytest.mark.parametrize("split", [0, 1024])
def test_copy_ring_output_only_8_byte_aligned(gpu, split):
    """The copy ring stores its output rows 16 bytes per lane; an output view
    that is only 8-byte aligned (head stride 132 elements, 4-element offset)
    takes its 8-byte store path and holds the same values as a contiguous
    output, for unsplit rows and for rows merged from split partials."""
    cfg = W.PrefillConfig("t", 2, 8, 2, 128, 32, 200, 0, 2500, seed=93)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    T = b.q.shape[0]
    wide = torch.full((T, cfg.q_heads, 136), 7.0, dtype=torch.bfloat16, device=gpu)
    view = wide[:, :, 4:132]
    assert view.data_ptr() % 16 == 8 and view.stride(1) == 136
    run = lambda out: K.paged_prefill(b.q, b.cu_seqlens, b.prior, b.max_seqlen_q, b.k_cache,
                                      b.v_cache, b.block_table, scale=cfg.head_dim ** -0.5,
                                      split_tokens=split, out=out)
    base = run(None)
    run(view)
    torch.cuda.synchronize()
    assert torch.equal(view, base)
    assert (wide[:, :, :4] == 7.0).all() and (wide[:, :, 132:] == 7.0).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bs,new,prior,window,use_sink", [
    (16, 1, 0, 0, False),        # one row, one key
    (32, 63, 0, 0, True),        # one partial key tile
    (64, 64, 64, 0, False),      # rows and keys end on a tile
    (16, 65, 192, 0, False),     # one key past a tile, the row tile wraps
    (128, 129, 128, 64, True),   # block wider than a tile, window edge inside one
    (16, 200, 320, 130, False),
])
def test_copy_ring_tile_edges_and_rising_scores(gpu, d, bs, new, prior, window, use_sink):
    """Row and key counts at the edges of the tiles, with scores that rise by
    far more than 2^8 between key tiles, so that every row's maximum moves
    several times.  Score error: q * scale is rounded to bf16 (relative 2^-9,
    uniform: rms 2^-9 / sqrt 3), which moves a score of standard deviation 4
    by 4.5e-3 rms, four times that at the tail; it enters the output as a
    relative error of the probabilities, on top of the 2e-2 that the bf16
    probabilities and output are allowed."""
    cfg = W.PrefillConfig("t", 1, 8, 2, d, bs, new, prior, prior, seed=140 + new)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    n = prior + new
    for t in range(n):  # keys of tile t / 64: standard deviation 0.25, 1, 4, 4, ...
        blk = int(b.block_table[0, t // bs])
        b.k_cache[blk, :, t % bs] *= min(4.0, 0.25 * 4.0 ** (t // 64))
    sink = torch.randn(8, generator=torch.Generator().manual_seed(new)).to(gpu) if use_sink else None
    out = K.paged_prefill(b.q, b.cu_seqlens, b.prior, new, b.k_cache, b.v_cache, b.block_table,
                          scale=d ** -0.5, sliding_window=window, sink=sink)
    ks = _seq_kv(b.k_cache.cpu(), b.block_table[0].cpu(), n, 2)
    vs = _seq_kv(b.v_cache.cpu(), b.block_table[0].cpu(), n, 2)
    f = OSg.fp32_prefill(b.q.cpu(), ks, vs, prior, d ** -0.5, window,
                         None if sink is None else sink.cpu())
    err = (out.float().cpu().double() - f).abs().max().item()
    assert err <= TOL_BF16 + 4 * 4.5e-3, err


EVEN_CASES = [
    # q heads, kv heads, d, bs, new, prior, table tokens, window, sink, fp8, rows cut, chunks
    (8, 2, 128, 32, 1, 4096, 0, 0, False, False, 4, 16),      # one row, 4-wave workgroups
    (32, 8, 128, 16, 200, 5000 // 16 * 16, 0, 0, True, False, 800, 6),   # 4-wave, 6 chunks
    (32, 8, 128, 32, 500, 8800, 0, 0, True, False, 2000, 4),  # 8-wave, 4 chunks
    (32, 8, 128, 32, 65, 640, 16384, 0, True, False, 260, 12),  # table far wider than the sequence
    (64, 8, 64, 32, 400, 288, 131072, 0, True, False, 3200, 12),  # the same, 8-wave, d = 64
    (8, 1, 64, 64, 33, 9600, 0, 0, True, False, 264, 32),     # 32 chunks, one kv head
    (64, 8, 64, 32, 1100, 4096, 0, 0, True, False, 768, 6),   # whole rounds of uncut row tiles
    (32, 8, 64, 16, 130, 6000 // 16 * 16, 0, 1500, False, False, 520, 4),  # window cut across chunks
    (12, 2, 128, 64, 100, 4096, 0, 0, False, True, 600, 16),  # FP8 ring
    (12, 2, 64, 64, 100, 4096, 0, 0, True, True, 600, 16),    # FP8, register-staged kernel
    (48, 8, 128, 64, 1536, 1088, 16384, 0, False, True, 1024, 6),  # FP8, 4 of 36 row tiles cut
]


@pytest.mark.parametrize("case", range(len(EVEN_CASES)))
def test_single_sequence_even_split(gpu, case):
    """One sequence whose row tiles are cut evenly on the device: equal to the
    uncut launch within two bf16 steps (each chunk keeps its own running
    maximum; partials are fp32), and within tolerance of float64 math."""
    Hq, Hkv, d, bs, new, prior, wide, win, use_sink, fp8, rows, chunks = EVEN_CASES[case]
    cfg = W.PrefillConfig("e", 1, Hq, Hkv, d, bs, new, prior, prior, fp8=fp8, seed=170 + case)
    b = W.make_prefill_batch(cfg, gpu)
    kw = {}
    if fp8:
        kw = dict(k_dequant=b.k_dequant, v_dequant=b.v_dequant)
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache, quant_mode=2,
                   k_scale=b.k_quant, v_scale=b.v_quant, scale_per_head=True)
    else:
        K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    table = b.block_table
    if wide:
        table = torch.full((1, wide // bs), -1, dtype=torch.int32, device=gpu)
        table[:, :b.block_table.shape[1]] = b.block_table
    keys = table.shape[1] * bs
    assert workspace_bytes(Hq, Hkv, d, bs, new, keys, fp8, win) == even_bytes(Hkv, d, rows, chunks)
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(case)).to(gpu) if use_sink else None
    run = lambda split: K.paged_prefill(b.q, b.cu_seqlens, b.prior, new, b.k_cache, b.v_cache, table,
                                        scale=d ** -0.5, sliding_window=win, sink=sink,
                                        split_tokens=split, **kw)
    got, base = run(0), run(1 << 20)
    assert (got.float() - base.float()).abs().max().item() <= 1.6e-2
    n, first = prior + new, max(0, new - 40)  # float64 on the last rows
    kc, vc = b.k_cache.cpu(), b.v_cache.cpu()
    if fp8:
        kc = kc.float() * b.k_dequant.cpu().view(1, -1, 1, 1)
        vc = vc.float() * b.v_dequant.cpu().view(1, -1, 1, 1)
    ks, vs = (_seq_kv(c, b.block_table[0].cpu(), n, Hkv) for c in (kc, vc))
    f = OSg.fp32_prefill(b.q[first:].cpu(), ks, vs, prior + first, d ** -0.5, win,
                         None if sink is None else sink.cpu())
    err = (got[first:].float().cpu().double() - f).abs().max().item()
    assert err <= (TOL_FP8 if fp8 else TOL_BF16), err


def test_single_sequence_without_workspace(gpu):
    """The C entry with no workspace runs a short single sequence unsplit
    (the wrapper would allocate one for the even split)."""
    import ctypes

    from vllm_neuron_amd import _native as N

    cfg = W.PrefillConfig("t", 1, 8, 2, 128, 32, 64, 2048, 2048, seed=7)
    b = W.make_prefill_batch(cfg, gpu)
    K.kv_write(b.k_new, b.v_new, b.slots, b.k_cache, b.v_cache)
    base = K.paged_prefill(b.q, b.cu_seqlens, b.prior, 64, b.k_cache, b.v_cache, b.block_table,
                           scale=0.1, split_tokens=1 << 20)
    out = torch.zeros_like(base)
    a = N.PrefillArgs()
    a.q, a.q_stride = b.q.data_ptr(), tuple(b.q.stride())
    a.num_seqs, a.max_seqlen_q, a.num_tokens = 1, 64, 64
    a.cu_seqlens_q, a.prior_tokens = b.cu_seqlens.data_ptr(), b.prior.data_ptr()
    a.k_cache, a.v_cache = b.k_cache.data_ptr(), b.v_cache.data_ptr()
    a.cache_dtype = a.out_dtype = N.DTYPE_BF16
    a.k_cache_stride, a.v_cache_stride = (*b.k_cache.stride(), 0), tuple(b.v_cache.stride())
    a.num_blocks, a.block_size = b.k_cache.shape[0], 32
    a.block_table, a.blocks_per_seq = b.block_table.data_ptr(), b.block_table.shape[1]
    a.bt_stride = (b.block_table.stride(0), 0, 1)
    a.num_q_heads, a.num_kv_heads, a.head_dim, a.scale = 8, 2, 128, 0.1
    a.out, a.out_stride = out.data_ptr(), tuple(out.stride())
    assert N.lib().mia_prefill_workspace_bytes(ctypes.byref(a)) > 0
    N.check(N.lib().mia_paged_prefill(ctypes.byref(a), N.stream_ptr(gpu)), "paged_prefill")
    assert torch.equal(out, base)


def _cache_of(rows, bs, dtype, gpu, packed=False):
    """Block cache ``[1 + n / bs, 1, bs, d]`` (null block 0) and table of one
    sequence from its rows ``[n, d]``."""
    n, d = rows.shape
    c = torch.zeros(1 + n // bs, 1, bs, d)
    c[1:, 0] = rows.view(n // bs, bs, d)
    return c.to(dtype).to(gpu), torch.arange(1, 1 + n // bs, dtype=torch.int32, device=gpu)[None]


@pytest.mark.parametrize("d, bs, dtype, compact", [
    (64, 32, torch.bfloat16, False),   # copy ring
    (64, 4, torch.bfloat16, False),    # register-staged
    (128, 32, torch.bfloat16, False),  # copy ring
    (128, 32, torch.bfloat16, True),   # four waves, tested by the maximum
    (128, 4, torch.bfloat16, False),
    (128, 32, torch.float8_e4m3fn, False),
    (64, 32, torch.float8_e4m3fn, False),
])
def test_maximum_moves_past_8_only(gpu, d, bs, dtype, compact):
    """The running maximum moves when a score passes it by more than 8 (log2
    units), whatever the tile's sum is: one key of score 0, then 64 keys of
    score 5.34375 whose V is 0.  Their weights 2^5.34375 = 40.61 are rounded to
    bf16 (40.5), so a channel of the first key's V comes out as v / (1 + 64 *
    40.5); a maximum moved to 5.34375 would give v / (1 + 64 * 40.61)."""
    n = 128
    k = torch.zeros(n, d)
    k[1:64, 2] = -192.0  # no weight
    k[64:, 0], k[64:, 1] = 5.0, 0.34375
    v = torch.zeros(n, d)
    ch = torch.arange(d)
    v[0] = (8 + ch % 8) / 8.0 * 2.0 ** (ch // 8 % 4)
    kc, table = _cache_of(k, bs, dtype, gpu)
    vc, _ = _cache_of(v, bs, dtype, gpu)
    q = torch.zeros(1, 1, d, dtype=torch.bfloat16, device=gpu)
    q[0, 0, :3] = 1.0
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)
    out = K.paged_prefill(q, i32([0, 1]), i32([n - 1]), 1, kc, vc, table,
                          scale=0.6931471805599453, compact_kernel=compact)
    got = out[0, 0].double().cpu()
    want = (v[0].double() / (1 + 64 * 40.5))
    moved = (v[0].double() / (1 + 64 * 2.0 ** 5.34375)).to(torch.bfloat16).double()
    # half a bf16 step is 2^-9 relative at most; the fp32 steps add some 2^-22
    assert bool(((got - want).abs() <= want * (2.0 ** -8)).all())
    bits = want.to(torch.bfloat16).double()
    assert int((bits != moved).sum()) >= d // 8  # the two rules are told apart
    assert torch.equal(got, bits)


@pytest.mark.parametrize("Hq, Hkv, d, bs, fp8, packed, new, prior, window, compact", [
    (8, 2, 64, 32, False, False, 100, 41, 0, False),     # copy ring: keys end inside a block
    (8, 2, 64, 16, False, False, 70, 129, 0, False),     # and a table entry of -1 inside the tile
    (8, 2, 64, 16, False, False, 200, 1000, 128, False),  # freed blocks before the window
    (8, 2, 64, 4, False, False, 100, 41, 50, False),     # register-staged
    (8, 2, 64, 32, False, False, 65, 5000, 0, False),    # chunks of an even split
    (8, 2, 128, 32, False, False, 100, 41, 0, False),
    (8, 2, 128, 16, False, False, 200, 1000, 128, False),
    (8, 2, 128, 32, False, False, 300, 500, 0, True),    # two-stage ring
    (8, 2, 128, 128, False, False, 1, 0, 0, False),      # a single key
    (8, 2, 128, 64, True, False, 100, 41, 0, False),
    (8, 2, 128, 64, True, True, 90, 1000, 128, False),
    (8, 2, 64, 32, True, False, 100, 41, 33, False),
])
def test_unattended_cache_slots_do_not_matter(gpu, Hq, Hkv, d, bs, fp8, packed, new, prior, window,
                                              compact):
    """Slots that no row sees (past the last key, of the null block, of blocks
    freed before the window) may hold NaN: the outputs are those over a cache
    that holds zeros there, bit for bit."""
    g = torch.Generator().manual_seed(91)
    n = prior + new
    used = -(-n // bs)
    first = max(0, prior - window + 1) // bs if window else 0  # blocks before it are freed
    table = torch.full((1, used + 7), -1, dtype=torch.int32)
    table[0, :used] = 1 + torch.randperm(used, generator=g).to(torch.int32)
    table[0, :first] = 0
    dt = torch.float8_e4m3fn if fp8 else torch.bfloat16

    def cache(rows, fill):
        c = torch.full((used + 2, Hkv, bs, d), fill)
        for j in range(first, used):
            m = min(bs, n - j * bs)
            c[table[0, j], :, :m] = rows[:, j * bs:j * bs + m]
        return c.to(dt)

    def pack(c):  # [nb, Hkv, bs, d] -> [nb, Hkv, bs / 2, d, 2]
        return c.view(torch.uint8).view(*c.shape[:2], bs // 2, 2, d).transpose(3, 4).contiguous().view(dt)

    kr, vr = (torch.randn(Hkv, n, d, generator=g) for _ in range(2))
    q = torch.randn(new, Hq, d, generator=g).to(torch.bfloat16).to(gpu)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=gpu)

    def run(fill):
        kc, vc = cache(kr, fill), cache(vr, fill)
        return K.paged_prefill(q, i32([0, new]), i32([prior]), new, (pack(kc) if packed else kc).to(gpu),
                               vc.to(gpu), table.to(gpu), scale=d ** -0.5, sliding_window=window,
                               k_packed=packed, compact_kernel=compact)

    clean, dirty = run(0.0), run(float("nan"))
    assert torch.isfinite(clean.float()).all()
    assert torch.equal(clean.view(torch.int16), dirty.view(torch.int16))
