"""Decode attention kernels and the decode schedule on an MI355X, through the C ABI, against the oracle."""
import pytest
import torch

from oracle import decode as ref

pytestmark = pytest.mark.gpu
D = 128
TOL_BF16 = 2e-2


def rel_err(got, want):
    got, want = got.double().cpu(), want.double().cpu()
    return ((got - want).abs().max() / want.abs().max().clamp_min(1e-30)).item()


@pytest.fixture(scope="module")
def ops():
    from dynaflow_amd import ops as _ops

    return _ops


def natural(k_cache, v_cache):
    """Product caches -> float64 [slots, capacity, kv_heads, d] on the host."""
    from dynaflow_amd.decode import unpack_v_cache

    return (k_cache.double().cpu().permute(0, 2, 1, 3).contiguous(),
            unpack_v_cache(v_cache).double().cpu().permute(0, 2, 1, 3).contiguous())


@pytest.mark.parametrize("heads,kv_heads,capacity,lengths", [
    (4, 1, 32, [1, 2, 31, 32]),
    (8, 2, 64, [33, 64, 1, 17, 40]),
    (32, 8, 256, [256, 129, 128, 127, 5, 200]),
    (16, 1, 96, [96, 95, 65]),            # 16 query heads on one kv head: every MFMA row in use
    (3, 3, 160, [160, 1, 77, 159]),       # no grouping
])
def test_decode_attention_against_oracle(ops, heads, kv_heads, capacity, lengths):
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    T, slots_n = len(lengths), len(lengths) + 2
    g = torch.Generator().manual_seed(capacity + heads)
    k_nat = torch.randn(slots_n, kv_heads, capacity, D, generator=g).bfloat16()
    v_nat = torch.randn(slots_n, kv_heads, capacity, D, generator=g).bfloat16()
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g).bfloat16()
    slots = torch.randperm(slots_n, generator=g)[:T].int()
    lens = torch.tensor(lengths, dtype=torch.int32)
    cos, sin = rope_tables(capacity, D, 500000.0)
    k_cache, v_cache = k_nat.cuda(), pack_v_cache(v_nat).cuda()
    out = ops.decode_attention(qkv.cuda(), k_cache, v_cache, slots.cuda(), lens.cuda(), cos.cuda(), sin.cuda(),
                               heads, kv_heads)
    torch.cuda.synchronize()
    # oracle: rotate in float64, append, attend
    pos = lens.long() - 1
    q = ref.rope_at(qkv[:, : heads * D].double().view(T, heads, D), pos, 500000.0)
    k_new = ref.rope_at(qkv[:, heads * D:(heads + kv_heads) * D].double().view(T, kv_heads, D), pos, 500000.0)
    v_new = qkv[:, (heads + kv_heads) * D:].double().view(T, kv_heads, D)
    kc, vc = k_nat.double().permute(0, 2, 1, 3).contiguous(), v_nat.double().permute(0, 2, 1, 3).contiguous()
    got_k, got_v = natural(k_cache, v_cache)
    for t in range(T):
        s, L = int(slots[t]), int(lens[t])
        kc[s, L - 1], vc[s, L - 1] = k_new[t], v_new[t]
        want = ref.attend(q[t], kc[s, :L], vc[s, :L]).reshape(-1)
        assert rel_err(out[t].float(), want) < TOL_BF16, (t, L)
    # the caches: new k within one bf16 rounding of the rotated value, new v bit-exact, everything else untouched
    assert (got_k - kc).abs().max() <= 2 ** -8 * kc.abs().max()
    assert torch.equal(got_v, vc)
    untouched = torch.ones(slots_n, capacity, dtype=torch.bool)
    untouched[slots.long(), pos] = False
    assert torch.equal(got_k[untouched], k_nat.double().permute(0, 2, 1, 3)[untouched])


def test_decode_attention_over_consecutive_steps_reads_what_the_previous_launch_appended(ops):
    """Four launches in a row on the same caches, every sequence one position further each time (crossing chunk
    boundaries of 32 and 8 positions): a launch attends over the keys and values that the launches before it
    appended - written by ordinary stores, read back by the next kernel's non-temporal loads."""
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    heads, kv_heads, capacity, start = 8, 2, 96, [1, 30, 31, 62, 7]
    T = len(start)
    g = torch.Generator().manual_seed(77)
    k_nat = torch.randn(T, kv_heads, capacity, D, generator=g).bfloat16()
    v_nat = torch.randn(T, kv_heads, capacity, D, generator=g).bfloat16()
    cos, sin = rope_tables(capacity, D, 500000.0)
    k_cache, v_cache = k_nat.cuda(), pack_v_cache(v_nat).cuda()
    kc, vc = k_nat.double().permute(0, 2, 1, 3).contiguous(), v_nat.double().permute(0, 2, 1, 3).contiguous()
    slots = torch.arange(T, dtype=torch.int32)
    for step in range(4):
        lens = torch.tensor([L + step for L in start], dtype=torch.int32)
        qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g).bfloat16()
        out = ops.decode_attention(qkv.cuda(), k_cache, v_cache, slots.cuda(), lens.cuda(), cos.cuda(), sin.cuda(),
                                   heads, kv_heads)
        pos = lens.long() - 1
        q = ref.rope_at(qkv[:, : heads * D].double().view(T, heads, D), pos, 500000.0)
        k_new = ref.rope_at(qkv[:, heads * D:(heads + kv_heads) * D].double().view(T, kv_heads, D), pos, 500000.0)
        v_new = qkv[:, (heads + kv_heads) * D:].double().view(T, kv_heads, D)
        for t in range(T):
            L = int(lens[t])
            # what the kernel left in the cache: the rotated key rounded to bf16, the value as it came
            kc[t, L - 1], vc[t, L - 1] = k_new[t].bfloat16().double(), v_new[t]
            want = ref.attend(q[t], kc[t, :L], vc[t, :L]).reshape(-1)
            assert rel_err(out[t].float(), want) < TOL_BF16, (step, t, L)
    got_k, got_v = natural(k_cache, v_cache)
    assert (got_k - kc).abs().max() <= 2 ** -7 * kc.abs().max()
    assert torch.equal(got_v, vc)


@pytest.mark.parametrize("heads,kv_heads,capacity,lengths", [
    (4, 1, 32, [1, 2, 31, 32, 40]),                  # 40: beyond the capacity, nothing is appended
    (32, 8, 256, [256, 129, 128, 127, 5, 200, 97]),
    (16, 1, 96, [96, 95, 65, 33, 8]),
    (3, 3, 160, [160, 1, 77, 159]),
])
def test_one_launch_decode_attention_has_the_bits_of_the_two_launches(heads, kv_heads, capacity, lengths):
    """dfhip_decode_attention_append_bf16 (rotation, cache append and attention in one launch) against
    dfhip_rope_kv_append_bf16 followed by dfhip_decode_attention_bf16 through the C ABI: the same output bits and
    the same caches, the new position in every place a fragment can hold it, a bad slot and a length beyond the
    capacity included."""
    import math

    from dynaflow_amd import _cabi
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    lib = _cabi.load()
    T, slots_n = len(lengths), len(lengths) + 2
    g = torch.Generator().manual_seed(7 * capacity + heads)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g).bfloat16().cuda()
    slots = torch.randperm(slots_n, generator=g)[:T].int()
    slots[-1] = slots_n + 3 if capacity == 160 else slots[-1]       # one token with a slot out of range
    slots = slots.cuda()
    lens = torch.tensor(lengths, dtype=torch.int32).cuda()
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    k0 = torch.randn(slots_n, kv_heads, capacity, D, generator=g).bfloat16()
    v0 = pack_v_cache(torch.randn(slots_n, kv_heads, capacity, D, generator=g).bfloat16())
    stream = torch.cuda.current_stream().cuda_stream
    scale = 1.0 / math.sqrt(D)

    k_two, v_two = k0.clone().cuda(), v0.clone().cuda()
    q_rot = torch.empty(T, heads * D, dtype=torch.bfloat16, device="cuda")
    out_two = torch.full((T, heads * D), 7.0, dtype=torch.bfloat16, device="cuda")
    print(f"two launches heads={heads} kv_heads={kv_heads} capacity={capacity}", flush=True)
    _cabi.check("dfhip_rope_kv_append_bf16", lib.dfhip_rope_kv_append_bf16(
        qkv.data_ptr(), qkv.stride(0), q_rot.data_ptr(), heads * D, k_two.data_ptr(), v_two.data_ptr(), slots.data_ptr(),
        lens.data_ptr(), cos.data_ptr(), sin.data_ptr(), T, heads, kv_heads, D, slots_n, capacity, cos.shape[0], stream))
    _cabi.check("dfhip_decode_attention_bf16", lib.dfhip_decode_attention_bf16(
        q_rot.data_ptr(), heads * D, k_two.data_ptr(), v_two.data_ptr(), slots.data_ptr(), lens.data_ptr(),
        out_two.data_ptr(), heads * D, T, heads, kv_heads, D, slots_n, capacity, scale, stream))
    k_one, v_one = k0.clone().cuda(), v0.clone().cuda()
    out_one = torch.full((T, heads * D), 7.0, dtype=torch.bfloat16, device="cuda")
    print("one launch", flush=True)
    _cabi.check("dfhip_decode_attention_append_bf16", lib.dfhip_decode_attention_append_bf16(
        qkv.data_ptr(), qkv.stride(0), k_one.data_ptr(), v_one.data_ptr(), slots.data_ptr(), lens.data_ptr(),
        cos.data_ptr(), sin.data_ptr(), out_one.data_ptr(), heads * D, T, heads, kv_heads, D, slots_n, capacity,
        cos.shape[0], scale, stream))
    torch.cuda.synchronize()
    assert torch.equal(k_one, k_two) and torch.equal(v_one, v_two)
    assert not torch.equal(k_one.cpu(), k0)                       # something was appended
    assert torch.equal(out_one, out_two)
    assert torch.isfinite(out_one.float()).all()


@pytest.mark.parametrize("heads,kv_heads,capacity,lengths", [
    (32, 8, 512, [1, 512, 33, 256]),                 # room for two parts, which do not pay: whole
    (4, 1, 8192, [8192, 1, 300]),                    # 32 parts for the long one, the short ones whole
    (16, 1, 4096, [4095, 2049, 7, 65]),              # 16 query heads on one kv head
    (3, 3, 1024, [1024, 31, 513] * 7),               # no grouping
    (32, 8, 2048, [2048 - 31 * i for i in range(32)]),   # two parts again
    (32, 8, 2048, [2048 - 64 * i for i in range(21)]),   # the most pairs that are still cut: three parts each
    (8, 2, 4096, [767, 768, 1023, 1024, 1025, 4096]),    # around the lengths that take one, three and four parts
    (32, 8, 4096, [4096, 1, 2500, 255]),             # 16 parts for the longest, nine, and two whole
    (3, 3, 4096, [4096 - 370 * i for i in range(11)]),   # fifteen parts and fewer
])
def test_decode_attention_cut_over_positions(ops, heads, kv_heads, capacity, lengths):
    """Few (token, kv head) pairs: several workgroups share a token's positions and the last to arrive combines them.
    Against the uncut launch of the same inputs (which the tests above hold to the oracle; two bf16 roundings of the
    output apart: 2^-7 of the largest value), the same caches, the same bits in every run and counters left at zero."""
    import math

    from dynaflow_amd import _cabi
    from dynaflow_amd.decoder import rope_tables

    lib = _cabi.load()
    T, slots_n = len(lengths), len(lengths) + 1
    assert lib.dfhip_decode_attention_workspace_bytes(T, heads, kv_heads, capacity) > 0
    g = torch.Generator(device="cuda").manual_seed(capacity)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g, device="cuda").bfloat16()
    slots = torch.randperm(slots_n, generator=g, device="cuda")[:T].int()
    lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    k0 = torch.randn(slots_n, kv_heads, capacity, D, generator=g, device="cuda").bfloat16()
    v0 = torch.randn(slots_n, kv_heads, capacity // 8, D, 8, generator=g, device="cuda").bfloat16()
    k1, v1 = k0.clone(), v0.clone()
    want = torch.empty(T, heads * D, dtype=torch.bfloat16, device="cuda")
    _cabi.check("append", lib.dfhip_decode_attention_append_bf16(
        qkv.data_ptr(), qkv.stride(0), k1.data_ptr(), v1.data_ptr(), slots.data_ptr(), lens.data_ptr(), cos.data_ptr(),
        sin.data_ptr(), want.data_ptr(), heads * D, T, heads, kv_heads, D, slots_n, capacity, capacity,
        1.0 / math.sqrt(D), torch.cuda.current_stream().cuda_stream))
    outs = []
    for _ in range(3):
        k2, v2 = k0.clone(), v0.clone()
        outs.append(ops.decode_attention(qkv, k2, v2, slots, lens, cos, sin, heads, kv_heads))
        assert torch.equal(k2, k1) and torch.equal(v2, v1)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert rel_err(outs[0], want) < 2 ** -7
    for ws in ops._attention_workspaces.values():
        assert int(ws[:4096].view(torch.int32).abs().sum()) == 0


@pytest.mark.parametrize("heads,kv_heads,capacity,lengths", [
    (32, 8, 2048, [2048 - 61 * i for i in range(33)]),   # the fewest and the most pairs of a little more than one per unit
    (32, 8, 2048, [767 + 31 * i for i in range(41)] + [1, 768, 4096, 2048, 1023, 33, 2017]),
    (43, 43, 4096, [4096, 1, 2500, 1024]),               # the fewest and the most pairs below one per unit
    (32, 8, 4096, [4096 - 171 * i for i in range(24)]),
])
def test_decode_attention_cut_in_four(ops, heads, kv_heads, capacity, lengths):
    """Pairs that would leave the compute units unevenly loaded."""
    from dynaflow_amd import _cabi

    T = len(lengths)
    counters, block = 4096, heads // kv_heads * (D // 4 + 1) * 16
    assert _cabi.load().dfhip_decode_attention_workspace_bytes(T, heads, kv_heads, capacity) == counters + T * kv_heads * 4 * block
    test_decode_attention_cut_over_positions(ops, heads, kv_heads, capacity, lengths)


@pytest.mark.parametrize("T,kv_heads,capacity", [
    (33, 8, 64), (64, 8, 64), (65, 4, 96), (256, 2, 32),       # longest first: one and four lengths a lane
    (257, 2, 32),                                             # the order of the tokens
    (20, 8, 4096), (36, 8, 2048), (86, 3, 2048),              # in parts: of eight heads together, of three one after the other
])
def test_decode_attention_in_any_order_of_the_sequences(ops, T, kv_heads, capacity):
    """More workgroups than compute units start with the longest sequences: every token gets its own result, wherever it stands
    in the batch, with many sequences of one length, some that are empty or longer than the cache, and slots that do not exist."""
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    g = torch.Generator().manual_seed(T + capacity)
    lens = torch.randint(1, capacity + 1, (T,), generator=g)
    lens[: T // 3] = lens[0]
    lens[T // 2], lens[T - 1], lens[T - 2], lens[1] = capacity, capacity + 5, 0, 1
    slots = torch.randperm(T, generator=g).int()
    slots[T // 4] = -1
    k_cache = torch.randn(T, kv_heads, capacity, D, generator=g).bfloat16().cuda()
    v_cache = pack_v_cache(torch.randn(T, kv_heads, capacity, D, generator=g).bfloat16()).cuda()
    qkv = torch.randn(T, 3 * kv_heads * D, generator=g).bfloat16()
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    lens = lens.int()

    def run(order):
        return ops.decode_attention(qkv[order].cuda(), k_cache, v_cache, slots[order].cuda(), lens[order].cuda(), cos, sin,
                                    kv_heads, kv_heads)

    straight, order = torch.arange(T), torch.randperm(T, generator=g)
    out = run(straight)
    assert torch.equal(run(order), out[order.cuda()])          # (the second launch appends what the first one did)
    kc, vc = (t.cuda() for t in natural(k_cache, v_cache))
    pos = (lens.long() - 1).clamp(0, capacity - 1)
    q = ref.rope_at(qkv[:, : kv_heads * D].double().view(T, kv_heads, D), pos, 500000.0).cuda()
    for t in range(T):
        s, L = int(slots[t]), min(int(lens[t]), capacity)
        want = ref.attend(q[t], kc[s, :L], vc[s, :L]).reshape(-1) if s >= 0 and L > 0 else torch.zeros(kv_heads * D)
        if int(lens[t]) <= capacity:                           # (beyond it the rotation is by the last angle of the table)
            assert rel_err(out[t].float(), want) < TOL_BF16, (t, L)


@pytest.mark.parametrize("T,capacity,lengths", [(2, 8192, [1, 33, 512, 767]), (8, 1024, [64, 767]), (32, 2048, [2048, 700])])
def test_decode_attention_stays_whole_where_parts_do_not_pay(ops, T, capacity, lengths):
    """Sequences too short for three parts of 256 positions, and launches with room for two parts only: the bits of the
    uncut launch."""
    from dynaflow_amd import _cabi
    from dynaflow_amd.decoder import rope_tables

    heads, kv_heads = 32, 8
    g = torch.Generator(device="cuda").manual_seed(T)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g, device="cuda").bfloat16()
    slots = torch.arange(T, dtype=torch.int32, device="cuda")
    lens = torch.tensor([lengths[i % len(lengths)] for i in range(T)], dtype=torch.int32, device="cuda")
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    k = torch.randn(T, kv_heads, capacity, D, generator=g, device="cuda").bfloat16()
    v = torch.randn(T, kv_heads, capacity // 8, D, 8, generator=g, device="cuda").bfloat16()
    k1, v1, want = k.clone(), v.clone(), torch.empty(T, heads * D, dtype=torch.bfloat16, device="cuda")
    _cabi.check("append", _cabi.load().dfhip_decode_attention_append_bf16(
        qkv.data_ptr(), qkv.stride(0), k1.data_ptr(), v1.data_ptr(), slots.data_ptr(), lens.data_ptr(), cos.data_ptr(),
        sin.data_ptr(), want.data_ptr(), heads * D, T, heads, kv_heads, D, T, capacity, capacity, D ** -0.5,
        torch.cuda.current_stream().cuda_stream))
    assert torch.equal(ops.decode_attention(qkv, k, v, slots, lens, cos, sin, heads, kv_heads), want)
    assert torch.equal(k, k1) and torch.equal(v, v1)


def test_decode_attention_cut_over_positions_keeps_nan(ops):
    """A part all of whose scores are NaN has no maximum, like a part without positions, and still reaches the output:
    one kv head's keys are NaN in whole parts (2, 3) of 256 positions; the other heads and tokens stay finite."""
    from dynaflow_amd.decoder import rope_tables

    T, heads, kv_heads, capacity = 2, 32, 8, 8192
    g = torch.Generator(device="cuda").manual_seed(5)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g, device="cuda").bfloat16()
    k = torch.randn(T, kv_heads, capacity, D, generator=g, device="cuda").bfloat16()
    v = torch.randn(T, kv_heads, capacity // 8, D, 8, generator=g, device="cuda").bfloat16()
    k[0, 3, 512:1024] = float("nan")
    slots, lens = (torch.tensor(t, dtype=torch.int32, device="cuda") for t in ([0, 1], [capacity, capacity]))
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    out = ops.decode_attention(qkv, k, v, slots, lens, cos, sin, heads, kv_heads).view(T, heads, D)
    want = torch.zeros(T, heads, D, dtype=torch.bool, device="cuda")
    want[0, 12:16] = True
    assert torch.equal(out.isnan(), want)


def test_decode_attention_ignores_what_lies_past_the_length(ops):
    """Caches are usually allocated uninitialised or hold recycled slots: NaN and Inf patterns in positions
    from lengths[t] on (keys and values) must not reach the output, and the result is the one a cache with
    zeros there gives, bit for bit."""
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    heads, kv_heads, capacity = 8, 2, 96
    lengths = [1, 7, 8, 31, 32, 33, 60, 96]
    T = len(lengths)
    g = torch.Generator().manual_seed(21)
    k_nat = torch.randn(T, kv_heads, capacity, D, generator=g).bfloat16()
    v_nat = torch.randn(T, kv_heads, capacity, D, generator=g).bfloat16()
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g).bfloat16()
    slots = torch.arange(T, dtype=torch.int32)
    lens = torch.tensor(lengths, dtype=torch.int32)
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    outs = []
    for junk in (0.0, float("nan"), float("inf")):
        k, v = k_nat.clone(), v_nat.clone()
        for t, L in enumerate(lengths):
            k[t, :, L:], v[t, :, L:] = junk, junk
        out = ops.decode_attention(qkv.cuda(), k.cuda(), pack_v_cache(v).cuda(), slots.cuda(), lens.cuda(), cos, sin,
                                   heads, kv_heads)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(out.float()).all()), junk
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_decode_attention_bad_slot_or_length_is_harmless(ops):
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    g = torch.Generator().manual_seed(1)
    k = torch.randn(2, 1, 32, D, generator=g).bfloat16().cuda()
    v = pack_v_cache(torch.randn(2, 1, 32, D, generator=g).bfloat16()).cuda()
    k0, v0 = k.clone(), v.clone()
    qkv = torch.randn(3, 6 * D, generator=g).bfloat16().cuda()
    cos, sin = rope_tables(32, D, 500000.0)
    out = ops.decode_attention(qkv, k, v, torch.tensor([5, -1, 1], dtype=torch.int32).cuda(),
                               torch.tensor([3, 3, 0], dtype=torch.int32).cuda(), cos.cuda(), sin.cuda(), 4, 1)
    torch.cuda.synchronize()
    assert torch.equal(out, torch.zeros_like(out)) and torch.equal(k, k0) and torch.equal(v, v0)


def test_decode_attention_full_size_properties(ops):
    """256 sequences x 2048 cached positions (the decode configuration): sampled tokens against the
    oracle, constant V gives that constant, run-to-run bit identity."""
    from dynaflow_amd.decoder import rope_tables

    T, heads, kv_heads, capacity = 256, 32, 8, 2048
    gen = torch.Generator(device="cuda").manual_seed(5)
    k_cache = torch.randn(T, kv_heads, capacity, D, generator=gen, device="cuda").bfloat16()
    v_cache = torch.randn(T, kv_heads, capacity // 8, D, 8, generator=gen, device="cuda").bfloat16()
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=gen, device="cuda").bfloat16()
    slots = torch.arange(T, dtype=torch.int32, device="cuda").flip(0).contiguous()
    lens = torch.full((T,), capacity, dtype=torch.int32, device="cuda")
    lens[::7] = 1500
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    out = ops.decode_attention(qkv, k_cache, v_cache, slots, lens, cos, sin, heads, kv_heads)
    again = ops.decode_attention(qkv, k_cache, v_cache, slots, lens, cos, sin, heads, kv_heads)
    torch.cuda.synchronize()
    assert torch.equal(out, again)
    kc, vc = None, None
    for t in (0, 7, 100, 255):
        s, L = int(slots[t]), int(lens[t])
        kn, vn = natural(k_cache[s:s + 1], v_cache[s:s + 1])
        pos = torch.tensor([L - 1])
        q = ref.rope_at(qkv[t:t + 1, : heads * D].double().cpu().view(1, heads, D), pos, 500000.0)[0]
        want = ref.attend(q, kn[0, :L], vn[0, :L]).reshape(-1)
        assert rel_err(out[t].float(), want) < TOL_BF16, t
    v_cache.fill_(0.375)
    qkv[:, (heads + kv_heads) * D:] = 0.375
    const = ops.decode_attention(qkv, k_cache, v_cache, slots, lens, cos, sin, heads, kv_heads)
    assert torch.equal(const, torch.full_like(const, 0.375))


def build_decode(T, whole_graph, sub_graphs=False, knobs=None, **over):
    from dynaflow_amd.backend import make_backend
    from dynaflow_amd.config import CUDAGraphConfig, DynaFlowConfig, InductorConfig
    from dynaflow_amd.decode import DecodeModel
    from dynaflow_amd.manager import DynaFlowManager

    cfg_model = dict(layers=3, vocab=500, hidden=512, heads=8, kv_heads=2, inter=1408, slots=T + 3, capacity=128)
    cfg_model.update(over)
    host = DecodeModel(**cfg_model, dtype=torch.bfloat16)
    host.init_weights(3)
    host.fill_caches(7)
    model = DecodeModel(**cfg_model, dtype=torch.bfloat16, device="cuda")
    model.load_state_dict(host.state_dict())
    for a, b in zip(model.attn, host.attn):
        a.k_cache.copy_(b.k_cache); a.v_cache.copy_(b.v_cache)
    g = torch.Generator().manual_seed(11)
    ids = torch.randint(0, cfg_model["vocab"], (T,), generator=g)
    slots = torch.randperm(cfg_model["slots"], generator=g)[:T].int()
    lengths = torch.randint(1, cfg_model["capacity"] + 1, (T,), generator=g).int()
    cfg = DynaFlowConfig("dynaflow_amd.schedulers:DecoderOverlapScheduler", 2, InductorConfig(enabled=True),
                         CUDAGraphConfig(enabled=sub_graphs, capture_sizes=[T // 2, T]),
                         {"min_nano_split_tokens": 1, "dump_graph": False, "whole_graph": whole_graph,
                          "max_tokens": T, **(knobs or {})})
    manager = DynaFlowManager()
    torch._dynamo.reset()
    dev = [t.cuda() for t in (ids, slots, lengths)]
    for t in dev:
        torch._dynamo.mark_dynamic(t, 0)
    compiled = torch.compile(model, backend=make_backend(manager, cfg), fullgraph=True)
    with torch.no_grad():
        manager.prepare(T, [1] * T)
        compiled(*dev)
    return manager, compiled, dev, host, model, (ids, slots, lengths), cfg_model


def test_decode_schedule_against_oracle():
    """Three layers, 24 sequences, two nano-batches on two streams: every sub-graph runs on HIP operators
    (attention sub-graphs on the main stream, MLP sub-graphs on the side stream) and the result matches the
    float64 oracle, as do the appended cache entries."""
    from dynaflow_amd import ops

    T = 24
    print("decode schedule: build (trace, lower, first call on the fast path)", flush=True)
    manager, compiled, dev, host, model, (ids, slots, lengths), cm = build_decode(T, whole_graph=False)
    subs = [n.target for n in manager.graph_module.graph.nodes if n.op == "call_module"]
    assert len(subs) == 6
    attn_targets = [n.target for n in manager.graph_module.__dict__[subs[0]].callable_dynamic.graph.nodes
                    if n.op == "call_function"]
    assert ops.decode_attention in attn_targets and ops.rms_norm in attn_targets
    assert attn_targets.count(ops.linear) == 1
    assert attn_targets.count(ops.linear_add) + attn_targets.count(ops.linear_add_to_output) == 1
    params = ref.params_of(host)
    kc, vc = ref.caches_of(host)
    want = ref.decode_step(ids, slots, lengths, params, kc, vc, cm["heads"], cm["kv_heads"])
    with torch.no_grad():
        print("decode schedule: eager two-stream run", flush=True)
        split = manager.prepare(T, [1] * T, use_cudagraph=False)
        y = compiled(*dev).clone()
        torch.cuda.synchronize()
        assert split.split_indices == [0, 12, 24]
        assert rel_err(y.float(), want) < TOL_BF16
        again = compiled_again(manager, compiled, dev, T)      # a decode step with fixed lengths is idempotent
        assert torch.equal(again, y)
    trace = manager.engine.issue_trace
    assert trace[:3] == [(subs[0], 0), (subs[1], 0), (subs[0], 1)] and len(trace) == 12
    for i, blk in enumerate(model.attn):
        got_k = blk.k_cache.double().cpu().permute(0, 2, 1, 3)
        assert (got_k - kc[i]).abs().max() <= 0.05 * kc[i].abs().max()


def compiled_again(manager, compiled, dev, T):
    manager.prepare(T, [1] * T, use_cudagraph=False)
    out = compiled(*dev)
    torch.cuda.synchronize()
    return out


def test_decode_attention_under_graph_capture(ops):
    """The entry points allocate nothing and synchronise nothing, so the operator can be captured into a
    hipGraph: every replay (with eager work between replays) must equal the eager result, and a replay picks
    up new contents of the captured tensors."""
    from dynaflow_amd.decode import pack_v_cache
    from dynaflow_amd.decoder import rope_tables

    T, heads, kv_heads, capacity = 12, 8, 2, 128
    g = torch.Generator().manual_seed(2)
    k_cache = torch.randn(T + 3, kv_heads, capacity, D, generator=g).bfloat16().cuda()
    v_cache = pack_v_cache(torch.randn(T + 3, kv_heads, capacity, D, generator=g).bfloat16()).cuda()
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D, generator=g).bfloat16().cuda()
    slots = torch.randperm(T + 3, generator=g)[:T].int().cuda()
    lens = torch.randint(1, capacity + 1, (T,), generator=g).int().cuda()
    cos, sin = (t.cuda() for t in rope_tables(capacity, D, 500000.0))
    print("decode attention: eager", flush=True)
    eager = ops.decode_attention(qkv, k_cache, v_cache, slots, lens, cos, sin, heads, kv_heads).clone()
    torch.cuda.synchronize()
    print("decode attention: capture", flush=True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.decode_attention(qkv, k_cache, v_cache, slots, lens, cos, sin, heads, kv_heads)
    for i in range(3):
        print(f"decode attention: replay {i}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"replay {i}"
        torch.randn(256, 256, device="cuda").sum().item()
    qkv.copy_(torch.randn(qkv.shape, generator=g).bfloat16())
    graph.replay()
    torch.cuda.synchronize()
    want = ops.decode_attention(qkv, k_cache, v_cache, slots, lens, cos, sin, heads, kv_heads)
    assert torch.equal(out, want) and not torch.equal(out, eager)


@pytest.mark.parametrize("streams,share", [("by_kind", 1), ("by_nano_batch", 1), ("by_nano_batch", 2)])
def test_decode_schedule_with_sub_graph_replay(streams, share):
    """Per-sub-graph graphs (the reference's mechanism) on the decode model at shapes where the projections
    run on the weight-streaming kernel with K split: capture in a dry-run at the nano-batch size, then the
    scheduled forward replays the graphs; every replay equals the eager two-stream result - with the streams
    chosen by sub-graph kind (attention / MLP), with one stream per nano-batch, and with the kernels planned
    for two launches that share the GPU (knob side_by_side: K split over fewer workgroups)."""
    T = 32
    over = dict(layers=2, hidden=1024, heads=8, kv_heads=2, inter=2048)
    print("decode sub-graph replay: eager model", flush=True)
    manager, compiled, dev, host, model, inputs, cm = build_decode(T, whole_graph=False,
                                                                   knobs={"streams": streams, "side_by_side": share},
                                                                   **over)
    with torch.no_grad():
        manager.prepare(T, [1] * T)
        eager = compiled(*dev).clone()
        torch.cuda.synchronize()
    print("decode sub-graph replay: graph model", flush=True)
    manager, compiled, dev, host2, model2, _, _ = build_decode(T, whole_graph=False, sub_graphs=True,
                                                               knobs={"streams": streams, "side_by_side": share},
                                                               **over)
    half = T // 2
    with torch.no_grad():
        print("decode sub-graph replay: dry-run capture", flush=True)
        manager.prepare(half, [1] * half, is_dryrun=True, use_cudagraph=True)
        compiled(*(t[:half].contiguous() for t in dev))
        torch.cuda.synchronize()
        for i in range(3):
            print(f"decode sub-graph replay: replay {i}", flush=True)
            split = manager.prepare(T, [1] * T, use_cudagraph=True)
            assert split.use_cudagraph and split.num_tokens_padded == [half, half]
            y = compiled(*dev)
            torch.cuda.synchronize()
            assert torch.equal(y, eager), f"replay {i}"
            torch.randn(256, 256, device="cuda").sum().item()
    names = [n.target for n in manager.graph_module.graph.nodes if n.op == "call_module"]
    wrapper = manager.graph_module.__dict__[names[0]].callable_dynamic
    assert sorted(k[:2] for k in wrapper._entries) == [(half, 0), (half, 1)]


class _LayerwiseParams(dict):
    """``oracle.decode.params_of`` one tensor at a time: float64 copies are made when the oracle asks for them
    and not kept, so that a 32-layer model never sits on the host in float64 as a whole."""

    def __init__(self, model, embed_rows):
        super().__init__()
        self.model = model
        self.embed_rows = embed_rows                # the embedding rows of the sampled tokens, in their order

    def __getitem__(self, name):
        if name == "embed":
            return self.embed_rows
        kind, i = name.rsplit(".", 1)
        a, m = self.model.attn[int(i)], self.model.mlp[int(i)]
        t = {"attn_norm": a.norm_weight, "wqkv": a.wqkv, "wo": a.wo, "mlp_norm": m.norm_weight,
             "w_gate": m.w_gate, "w_up": m.w_up, "w_down": m.w_down}[kind]
        return t.detach().double().cpu()


def test_config4_full_size_properties():
    """The decode configuration at its real size: 32 Llama-3-8B-shaped layers, 256 single-token queries, 2048
    cached positions each (~N(0,1)), two nano-batches of 128.
    (1) ONE LAYER'S ARITHMETIC AT THE STATED TOLERANCE, for every layer: the float64 oracle runs the sampled tokens
    through the 32 layers; layer i of the HIP path (the same split schedule and kernels, a one-layer model that is
    given layer i's weights and caches) is fed the oracle's own input of that layer rounded to bf16 and must
    reproduce the oracle's output of that layer for that input within 2e-2.
    (2) end to end the bf16 roundings of the residual stream add up over 32 layers, so the distance of the whole
    step from the oracle is bounded relative to what eager PyTorch in bf16 - the reference implementation of the
    arithmetic - loses against the same oracle (not further than 1.5 x that, or 2e-2), and the HIP path may not be
    further from eager PyTorch than 1.5 x that either.
    (3) the split schedule against the same step as one batch through the same kernels, (4) run-to-run bit
    identity, (5) the whole split schedule replayed as ONE hipGraph has the bits of the eager schedule."""
    from dynaflow_amd.backend import make_backend
    from dynaflow_amd.config import CUDAGraphConfig, DynaFlowConfig, InductorConfig
    from dynaflow_amd.decode import DecodeModel
    from dynaflow_amd.manager import DynaFlowManager, trivial_split

    layers, seqs, capacity, heads, kv_heads = 32, 256, 2048, 32, 8
    print("config 4: build the model on the GPU", flush=True)
    model = DecodeModel(layers=layers, slots=seqs, capacity=capacity, dtype=torch.bfloat16, device="cuda")
    model.init_weights(0)
    model.fill_caches(5)
    gen = torch.Generator().manual_seed(4)
    ids = torch.randint(0, 128256, (seqs,), generator=gen)
    slots = torch.randperm(seqs, generator=gen).int()
    lengths = torch.full((seqs,), capacity, dtype=torch.int32)
    lengths[::5] = 1777                               # ragged: a last chunk of 17 positions
    lengths[3::11] = 1
    sampled = [0, 3, 127, 128, 255]
    # the sampled sequences' caches as they are before the step, natural layout, float64, on the host
    rows = slots[sampled].long().cuda()
    kc, vc = [], []
    for a in model.attn:
        k_nat, v_nat = natural(a.k_cache[rows], a.v_cache[rows])
        kc.append(k_nat)
        vc.append(v_nat)
    cfg = DynaFlowConfig("dynaflow_amd.schedulers:DecoderOverlapScheduler", 2, InductorConfig(enabled=True),
                         CUDAGraphConfig(enabled=False, capture_sizes=[seqs // 2, seqs]),
                         {"min_nano_split_tokens": 1, "dump_graph": False, "max_tokens": seqs,
                          "fuse_silu_epilogue": True, "whole_graph": True, "streams": "by_nano_batch"})
    manager = DynaFlowManager()
    torch._dynamo.reset()
    dev = [t.cuda() for t in (ids, slots, lengths)]
    for t in dev:
        torch._dynamo.mark_dynamic(t, 0)
    compiled = torch.compile(model, backend=make_backend(manager, cfg), fullgraph=True)
    with torch.no_grad():
        print("config 4: trace and first call", flush=True)
        manager.prepare(seqs, [1] * seqs)
        compiled(*dev)
        print("config 4: eager two-stream step", flush=True)
        split = manager.prepare(seqs, [1] * seqs, use_cudagraph=False)
        y = compiled(*dev).clone()
        torch.cuda.synchronize()
        assert split.split_indices == [0, 128, 256]
        assert len(manager.engine.issue_trace) == 2 * 2 * layers
        assert bool(torch.isfinite(y.float()).all())
        print("config 4: oracle on sampled tokens", flush=True)
        params = _LayerwiseParams(model, model.embed.detach()[ids[sampled].cuda()].double().cpu())
        n = len(sampled)
        lengths_s = lengths[sampled]
        twice_slots, twice_lengths = torch.arange(2 * n), torch.cat([lengths_s, lengths_s])
        # one pass over the layers gives both: the free-running oracle (rows 0 .. n-1) and, for the per-layer
        # check, each layer's output for the free-running input rounded to bf16 (rows n .. 2n-1, caches of their own)
        x_free = params["embed"][torch.arange(n)]
        forced_in, forced_want = [], []
        for i in range(layers):
            x_in = x_free.bfloat16().double()
            k2, v2 = torch.cat([kc[i], kc[i]]), torch.cat([vc[i], vc[i]])
            kc[i] = vc[i] = None
            out = ref.decode_layer(torch.cat([x_free, x_in]), twice_slots, twice_lengths, params, i, k2, v2, heads,
                                   kv_heads)
            forced_in.append(x_in)
            forced_want.append(out[n:])
            x_free = out[:n]
            del k2, v2
        want = x_free
        err = rel_err(y[sampled].float(), want)
        print("config 4: the same step by eager PyTorch in bf16", flush=True)
        aten = model(*dev)
        torch.cuda.synchronize()
        err_aten = rel_err(aten[sampled].float(), want)
        err_hip_aten = rel_err(y.float(), aten.float())
        print(f"config 4: against the float64 oracle: HIP path {err:.4f}, eager PyTorch bf16 {err_aten:.4f}; "
              f"HIP path against eager PyTorch {err_hip_aten:.4f}", flush=True)
        assert err < max(TOL_BF16, 1.5 * err_aten)
        assert err < 0.1                                   # and never by more than a rounding effect
        assert err_hip_aten < max(TOL_BF16, 1.5 * err_aten)   # two bf16 runs of 32 layers, all 256 tokens
        del aten
        print("config 4: the step as one batch", flush=True)
        manager.override_split_config(trivial_split(seqs, [1] * seqs, False, False))
        whole = compiled(*dev).clone()
        torch.cuda.synchronize()
        # other kernels for 256 rows than for 128, so other roundings: two bf16 runs of 32 layers differ from each
        # other by about what each differs from the oracle
        assert rel_err(y.float(), whole.float()) < max(2 ** -5, 1.5 * err_aten)
        print("config 4: second eager step", flush=True)
        manager.prepare(seqs, [1] * seqs, use_cudagraph=False)
        assert torch.equal(compiled(*dev), y)
        for i in range(3):
            print(f"config 4: whole-schedule graph, forward {i}", flush=True)
            manager.prepare(seqs, [1] * seqs, use_cudagraph=True)
            out = compiled(*dev)
            torch.cuda.synchronize()
            assert torch.equal(out, y), f"replay {i}"
        assert len(manager._schedule_graphs) == 1

        # ---- (1) layer by layer, teacher-forced: a one-layer model through the same scheduler, split and kernels
        print("config 4: per-layer check against the oracle (teacher-forced)", flush=True)
        from dynaflow_amd import ops as hip_ops

        one = DecodeModel(layers=1, vocab=seqs, slots=seqs, capacity=capacity, dtype=torch.bfloat16, device="cuda")
        manager_one = DynaFlowManager()
        torch._dynamo.reset()
        one_inputs = [torch.arange(seqs).cuda(), dev[1], dev[2]]
        for t in one_inputs:
            torch._dynamo.mark_dynamic(t, 0)
        compiled_one = torch.compile(one, backend=make_backend(manager_one, cfg), fullgraph=True)
        one.init_weights(1)
        manager_one.prepare(seqs, [1] * seqs)    # trace and first call (the manager splits from the second call on)
        compiled_one(*one_inputs)
        filler = y.clone()                       # rows of the other tokens: any finite hidden states will do
        worst = 0.0
        for i in range(layers):
            a, m = model.attn[i], model.mlp[i]
            for dst, src in ((one.attn[0].norm_weight, a.norm_weight), (one.attn[0].wqkv, a.wqkv),
                             (one.attn[0].wo, a.wo), (one.mlp[0].norm_weight, m.norm_weight),
                             (one.mlp[0].w_gate, m.w_gate), (one.mlp[0].w_up, m.w_up), (one.mlp[0].w_down, m.w_down),
                             (one.attn[0].k_cache, a.k_cache), (one.attn[0].v_cache, a.v_cache)):
                dst.copy_(src)
            rows_in = filler.clone()
            rows_in[sampled] = forced_in[i].to(torch.bfloat16).cuda()
            one.embed.copy_(rows_in)
            hip_ops.invalidate_stacked_weights()          # parameters were rewritten in place
            split = manager_one.prepare(seqs, [1] * seqs, use_cudagraph=False)
            got = compiled_one(*one_inputs)
            torch.cuda.synchronize()
            assert split.split_indices == [0, 128, 256]
            e = rel_err(got[sampled].float(), forced_want[i])
            worst = max(worst, e)
            assert e < TOL_BF16, f"layer {i}: {e:.4f} from the oracle's output for the same bf16 input"
        print(f"config 4: per-layer distance from the oracle, worst of {layers} layers: {worst:.5f}", flush=True)
