"""The launch plan of a single prefill sequence, read from the workspace that
the C entry asks for (256 CUs, with a GPU or without one)."""
import ctypes

import pytest

from vllm_neuron_amd import _native as N


def even_bytes(Hkv, d, cut_rows, chunks):
    """Partials of an even split: fp32 o, m, l and padding per row and chunk."""
    return Hkv * cut_rows * chunks * (4 * d + 16)


def prefill_args(Hq, Hkv, d, bs, new, table, fp8=False, window=0):
    """Arguments of one sequence over contiguous tensors (addresses made up)."""
    a = N.PrefillArgs()
    a.q = a.cu_seqlens_q = a.prior_tokens = a.k_cache = a.v_cache = a.block_table = a.out = 1 << 20
    a.q_stride = a.out_stride = (Hq * d, d, 1)
    a.num_seqs, a.max_seqlen_q, a.num_tokens = 1, new, new
    a.cache_dtype = N.DTYPE_FP8_E4M3FN if fp8 else N.DTYPE_BF16
    a.out_dtype = N.DTYPE_BF16
    a.k_cache_stride = (Hkv * bs * d, bs * d, d, 1, 0)
    a.v_cache_stride = (Hkv * bs * d, bs * d, d, 1)
    a.num_blocks, a.block_size, a.blocks_per_seq = table // bs + 1, bs, table // bs
    a.bt_stride = (table // bs, 0, 1)
    a.num_q_heads, a.num_kv_heads, a.head_dim, a.scale = Hq, Hkv, d, 0.1
    a.sliding_window = window
    return a


def workspace_bytes(*shape, **kw):
    n = N.lib().mia_prefill_workspace_bytes(ctypes.byref(prefill_args(*shape, **kw)))
    err = N.lib().mia_last_error()
    assert not err, err.decode()
    return n


@pytest.mark.parametrize("shape, cut_rows, chunks", [
    # 36 row tiles of 256 rows, 32 of them uncut: partials of the other 4 only
    (dict(Hq=48, Hkv=8, d=128, bs=64, new=1536, table=16384, fp8=True), 1024, 6),
    # 35 row tiles, 32 uncut; the last one is short
    (dict(Hq=64, Hkv=8, d=64, bs=32, new=1100, table=5216), 768, 6),
    # every row tile cut
    (dict(Hq=32, Hkv=8, d=128, bs=16, new=200, table=5200), 800, 6),
    (dict(Hq=8, Hkv=1, d=128, bs=64, new=33, table=9664), 264, 32),
])
def test_even_split_workspace_holds_the_cut_rows(shape, cut_rows, chunks):
    got = workspace_bytes(**shape)
    assert got == even_bytes(shape["Hkv"], shape["d"], cut_rows, chunks)


@pytest.mark.parametrize("new", [1, 64, 200, 777, 1100, 1500, 2048, 4096])
@pytest.mark.parametrize("table", [2048, 32768, 262144])
@pytest.mark.parametrize("Hq, Hkv, d, fp8", [(32, 8, 128, False), (8, 1, 128, False), (64, 8, 64, False),
                                             (48, 8, 128, True)])
def test_even_split_workspace_is_bounded(new, table, Hq, Hkv, d, fp8):
    """Under any table, a split takes at most 160 MiB of fp32 partials, or two
    bf16 halves (2 d + 16 bytes a row)."""
    halves = 2 * Hkv * new * (Hq // Hkv) * (2 * d + 16)
    assert workspace_bytes(Hq, Hkv, d, 128, new, table, fp8) <= max(160 << 20, halves)


@pytest.mark.parametrize("used, ok", [(0, True), (8, True), (120, True), (128, True), (200, True),
                                      (-8, False), (-1, False), (4, False), (100, False), (127, False)])
def test_head_dim_used_is_checked(used, ok):
    """A width that the kernels cannot honour is refused: taken as the full
    128 channels, rows of 100 would be read and written past their end."""
    a = prefill_args(8, 2, 128, 32, 64, 2048)
    a.head_dim_used = used
    a.num_tokens = 0  # nothing is launched
    rc = N.lib().mia_paged_prefill(ctypes.byref(a), None)
    assert (rc == 0) == ok
    assert ok or b"head_dim_used" in N.lib().mia_last_error()


@pytest.mark.parametrize("d, fp8", [(64, False), (128, False), (128, True)])
@pytest.mark.parametrize("bs", [32, 256])
def test_large_token_strides_keep_64_bit_offsets(d, fp8, bs):
    """A view whose tokens lie so far apart that a block spans 2^31 bytes runs
    the register-staged kernel (64-bit offsets) and not the copy ring: its plan
    is that of other strides the ring does not take, below that the ring's."""
    def plan(k_tok, v_tok, split=0):
        a = prefill_args(32, 8, d, bs, 300, 8192, fp8)
        a.split_tokens = split
        a.k_cache_stride = (d, 0, k_tok, 1, 0)
        a.v_cache_stride = (d, 0, v_tok, 1)
        n = N.lib().mia_prefill_workspace_bytes(ctypes.byref(a))
        assert not N.lib().mia_last_error()
        return n

    far = (1 << 31) // ((1 if fp8 else 2) * max(bs, 64))
    near, staged = plan(far - 16, far - 16), plan(far - 16, far - 32)
    assert near != staged  # the two kernels are told apart
    assert plan(far, far) == staged
