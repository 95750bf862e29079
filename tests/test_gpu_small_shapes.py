"""Shapes at the edges of the kernels' dispatch: the smallest launches, remainders of tiles, and the sizes on both sides
of a rule that picks a kernel variant."""
import pytest
import torch

from noise_amd import _lib
from tests._util import log_case

pytestmark = pytest.mark.gpu
DEV = 'cuda'


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _dense(x, w, layout, members, T):
    y = torch.empty(members * T, w.shape[0], device=DEV, dtype=torch.bfloat16)
    wp = w
    if layout == _lib.LAYOUT_WTILE:
        wp = torch.empty_like(w)
        _lib.call('noise_weight_tiles', w.data_ptr(), w.shape[0], w.shape[1], wp.data_ptr(), _stream())
    _lib.call('noise_dense_bf16', x.data_ptr(), _lib.LAYOUT_ROWS, w.shape[1], w.shape[0], wp.data_ptr(), layout, members,
              T, y.data_ptr(), _stream())
    torch.cuda.synchronize()
    return y


@pytest.mark.parametrize('dout', [256, 512, 1536])
@pytest.mark.parametrize('members,T', [(1, 32), (3, 96), (8, 256)])
def test_weight_resident_product_from_both_weight_layouts(members, T, dout):
    """The weight-resident kernel (512 deep, whole 32-row blocks) holds the same fragments whether the weight comes row
    by row through LDS or from WTILE blocks: equal bits, one block per launch up to several per workgroup, and within
    bf16 rounding (half a step of an 8-bit significand: 2^-8 relative) plus the fp32 sum's 512 2^-24 of the terms of the fp64 product."""
    g = torch.Generator().manual_seed(31)
    log_case(f'weight-resident product members={members} T={T} 512->{dout}')
    x = torch.randn(members * T, 512, generator=g).bfloat16()
    w = (torch.randn(dout, 512, generator=g) / 22).bfloat16()
    rows = _dense(x.to(DEV), w.to(DEV), _lib.LAYOUT_ROWS, members, T)
    tiles = _dense(x.to(DEV), w.to(DEV), _lib.LAYOUT_WTILE, members, T)
    assert torch.equal(rows, tiles)
    xd, wd = x.double(), w.double()
    ref = xd @ wd.t()
    bound = 2 ** -8 * ref.abs() + 512 * 2 ** -24 * (xd.abs() @ wd.abs().t())
    assert ((rows.cpu().double() - ref).abs() <= bound).all()


def _members_on_tiles(T, din, dout, result, most=140000):
    """tile -> the fewest members of T rows whose product takes it, for every tile that the rule takes up to `most`
    rows."""
    out = {}
    for m in range(1, most // T + 1):
        out.setdefault(_lib.value('noise_gemm_tile', m * T, din, dout, result), m)
    return out


@pytest.mark.parametrize('out', ['f32', 'bf16', 'accumulate'])
@pytest.mark.parametrize('dout,din,T', [(512, 576, 1000), (640, 1088, 1000), (512, 2048, 250), (384, 2048, 250)])
def test_tile_configurations_of_the_linear_agree_bit_for_bit(dout, din, T, out):
    """The tile GEMM takes 64 x 64, 128 x 128 or the large tiles (256 x 256; 256 x 128 where the columns are no multiple
    of 256) by the shape. Every member's rows are the same bits whichever it takes: the fewest rows that take each
    tile, against a few members on 64 x 64 tiles. T = 1000 and 250 leave ragged last tiles and tiles that straddle
    members."""
    from noise_amd import ops
    result = _lib.RESULT_BF16 if out == 'bf16' else _lib.RESULT_F32
    on = _members_on_tiles(T, din, dout, result)
    large = _lib.TILE_256X128 if dout % 256 else _lib.TILE_256X256
    assert set(on) == {large, _lib.TILE_128X128, _lib.TILE_64X64} and on[_lib.TILE_64X64] == 1
    g = torch.Generator().manual_seed(32)
    P, few = max(on.values()), max(1, 1000 // T)
    assert _lib.value('noise_gemm_tile', few * T, din, dout, result) == _lib.TILE_64X64
    log_case(f'linear tile configurations {din}->{dout} T={T} {out}: members {on}')
    x = torch.randn(P, T, din, generator=g).bfloat16().to(DEV)
    w = (torch.randn(dout, din, generator=g) * din ** -0.5).bfloat16().to(DEV)
    a, b = torch.randn(P, dout, generator=g).to(DEV), torch.randn(P, din, generator=g).to(DEV)
    sign = (1e-2 * torch.randn(P, generator=g)).to(DEV)
    res = torch.randn(P, T, dout, generator=g).to(DEV) if out == 'accumulate' else None

    def run(lo, hi):
        kw = dict(out=res[lo:hi].clone(), accumulate=True) if out == 'accumulate' else \
            dict(out_dtype=torch.bfloat16 if out == 'bf16' else torch.float32)
        return ops.lowrank_linear(x[lo:hi], w, a[lo:hi], b[lo:hi], sign[lo:hi], **kw)
    for members in (on[large], on[_lib.TILE_128X128]):
        whole = run(0, members)
        for lo in (0, members // 2, members - few):
            assert torch.equal(run(lo, lo + few), whole[lo:lo + few]), (members, lo)


@pytest.mark.parametrize('dout', [384, 512])
@pytest.mark.parametrize('din', [128, 192, 256, 320, 1536])
def test_dense_depths_around_the_steady_loop_on_every_tile(din, dout):
    """The dense product runs k stages 1 .. din / 32 - 4 from its steady loop in pairs: none at 4 or 6 stages, one pair at
    8 and 10, 22 at 48, and each tile has its own number of loads in flight. The fewest rows that take each tile (the
    large ones from a depth of 192 or 256 on), ragged in every tile: within one bf16 step of x W^T, and the same bits as
    its last members on 64 x 64 tiles, from a WTILE weight, and from TILE16 rows."""
    from tests._util import tile16_index
    T = 240
    on = _members_on_tiles(T, din, dout, _lib.RESULT_BF16)
    large = _lib.TILE_256X128 if dout % 256 else _lib.TILE_256X256
    assert {_lib.TILE_128X128, _lib.TILE_64X64} <= set(on) and (large in on or din < (256 if dout % 256 else 192))
    g = torch.Generator(DEV).manual_seed(48)
    w = (torch.randn(dout, din, device=DEV, generator=g) * din ** -0.5).bfloat16()
    wt = torch.empty_like(w)
    _lib.call('noise_weight_tiles', w.data_ptr(), dout, din, wt.data_ptr(), _stream())

    def run(x, members, x_layout=_lib.LAYOUT_ROWS, weight=w, w_layout=_lib.LAYOUT_ROWS):
        y = torch.empty(members * T, dout, device=DEV, dtype=torch.bfloat16)
        _lib.call('noise_dense_bf16', x.data_ptr(), x_layout, din, dout, weight.data_ptr(), w_layout, members, T,
                  y.data_ptr(), _stream())
        torch.cuda.synchronize()
        return y
    for tile, members in on.items():
        log_case(f'dense depth {din}->{dout} on tile {tile}: {members} members of {T} rows')
        x = torch.randn(members * T, din, device=DEV, generator=g).bfloat16()
        y = run(x, members)
        ref = (x.float() @ w.float().t()).bfloat16().float()
        assert ((y.float() - ref).abs() <= ref.abs() * 2 ** -7 + 1e-6).all()
        assert torch.equal(run(x[-3 * T:], min(3, members)), y[-3 * T:])
        with torch.device(DEV):
            at = tile16_index(members * T, din).flatten()
        x16 = torch.empty_like(x)
        x16.view(-1)[at] = x.view(-1)
        assert torch.equal(run(x, members, weight=wt, w_layout=_lib.LAYOUT_WTILE), y)
        assert torch.equal(run(x16, members, _lib.LAYOUT_TILE16, wt, _lib.LAYOUT_WTILE), y)


@pytest.mark.parametrize('T', [256, 250])
@pytest.mark.parametrize('head', ['fp32', 'bf16', 'fp32_split'])
def test_tile_configurations_of_the_head_agree_bit_for_bit(head, T):
    """The same for the head's per-token losses: the fewest rows that take each of its three tiles, against members at
    either end and in the middle on 64 x 64 tiles, from tiled operands (T = 256) and row-major ones with straddling tiles
    (T = 250)."""
    from noise_amd.population import HEAD_FORMAT
    g = torch.Generator().manual_seed(33)
    V, fmt = 4096, HEAD_FORMAT[head]
    on = _members_on_tiles(T, {'bf16': 512, 'fp32': 1024, 'fp32_split': 1536}[head], V, _lib.RESULT_HEAD, 40000)
    assert set(on) == {_lib.TILE_256X256, _lib.TILE_128X128, _lib.TILE_64X64} and on[_lib.TILE_64X64] == 1
    P = max(on.values())
    log_case(f'head tile configurations {head} T={T}: members {on}')
    x = torch.randn(P * T, 512, generator=g).to(DEV)
    w = (torch.randn(V, 512, generator=g) * 0.05).to(DEV)
    op = w
    if head != 'fp32':
        op = torch.empty(V, 1536 if head == 'fp32_split' else 512, device=DEV, dtype=torch.bfloat16)
        _lib.call('noise_cast_bf16', w.data_ptr(), op.data_ptr(), w.numel(), 512 if head == 'fp32_split' else 0, _stream())
    a, b = torch.randn(P, V, generator=g).to(DEV), torch.randn(P, 512, generator=g).to(DEV)
    sign = (1e-2 * torch.randn(P, generator=g)).to(DEV)
    tgt = torch.randint(0, V, (T,), generator=g).to(DEV)

    def run(lo, hi):
        m = hi - lo
        n = _lib.size_query('noise_head_ce_workspace_size', m, T, V, fmt)
        ws, loss = torch.empty(n, device=DEV, dtype=torch.uint8), torch.empty(m * T, device=DEV)
        _lib.call('noise_head_ce', x[lo * T:].data_ptr(), 0, None, op.data_ptr(), V, fmt, a[lo:].data_ptr(),
                  b[lo:].data_ptr(), sign[lo:].data_ptr(), tgt.data_ptr(), 0, m, T, 0, _lib.CE_NONE, loss.data_ptr(),
                  None, ws.data_ptr(), n, None, 0, _stream())
        torch.cuda.synchronize()
        return loss
    for members in (on[_lib.TILE_256X256], on[_lib.TILE_128X128]):
        whole = run(0, members)
        for lo in (0, members // 2, members - 1):
            assert torch.equal(run(lo, lo + 1), whole[lo * T:(lo + 1) * T]), (members, lo)


@pytest.mark.parametrize('shared', ['q', 'k'])
@pytest.mark.parametrize('qk_norm', [0, 1])
@pytest.mark.parametrize('n', [3, 40])
def test_attention_on_shared_heads_equals_packed_rows(n, shared, qk_norm):
    """Attention on separate operands, one of q and k and the values stored once per batch row for every draw, is bit for
    bit the attention on packed q | k | v rows that hold a copy per member: 64 queries per workgroup (3 draws) and 128
    (40)."""
    g = torch.Generator().manual_seed(34)
    b, T, window = 2, 256, 100
    log_case(f'attention on shared heads: {n} draws, {shared} shared, qk_norm={qk_norm}')

    def heads(blocks):
        x = torch.randn(blocks * T, 8, 64, generator=g)
        return (x * torch.rsqrt(x.square().mean(-1, keepdim=True))).view(blocks * T, 512).bfloat16().to(DEV)
    own, fixed = heads(n * b), heads(b)
    v = torch.randn(b * T, 512, generator=g).bfloat16().half().to(DEV)
    q, k = ((fixed, b), (own, n * b)) if shared == 'q' else ((own, n * b), (fixed, b))
    y = torch.empty(n * b * T, 512, device=DEV, dtype=torch.bfloat16)
    _lib.call('noise_attention_heads', q[0].data_ptr(), q[1], k[0].data_ptr(), k[1], v.data_ptr(), b, n * b, T, window,
              qk_norm, _lib.QK_BF16, y.data_ptr(), None, None, 0, None, _stream())
    rows = torch.cat([t[0].repeat(n * b // t[1], 1) for t in (q, k, (v.view(torch.bfloat16), b))], 1).contiguous()
    ref = torch.empty_like(y)
    _lib.call('noise_attention', rows.data_ptr(), n * b, T, window, qk_norm, _lib.QK_BF16, None, 0, ref.data_ptr(), None,
              None, None, 0, _stream())
    torch.cuda.synchronize()
    assert torch.equal(y, ref)


def test_credit_attention_of_strided_misaligned_and_float_heads():
    """credit.attention reads contiguous aligned bf16 heads in place; transposed, offset and fp32 ones give the same."""
    from noise_amd import credit
    g = torch.Generator().manual_seed(35)
    B, T = 2, 128
    log_case('credit.attention of strided, misaligned and fp32 heads')
    q, k, v = (torch.randn(B, T, 8, 64, generator=g).bfloat16().to(DEV) for _ in range(3))
    ref = credit.attention(q, k, v, 50)

    def strided(t):
        return t.transpose(1, 2).contiguous().transpose(1, 2)

    def shifted(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    for f in (strided, shifted, torch.Tensor.float):
        assert torch.equal(credit.attention(f(q), f(k), f(v), 50), ref), f


@pytest.mark.parametrize('fmt,qk_norm', [(_lib.QK_F16_Q_LOG2, 1), (_lib.QK_BF16_V_BF16, 1), (_lib.QK_BF16, 1),
                                         (_lib.QK_F16, 1), (_lib.QK_BF16, 0), (_lib.QK_F16, 0)])
@pytest.mark.parametrize('T,window', [(128, 128), (384, 65), (1152, 1100)])
def test_attention_of_64_and_128_queries_per_workgroup_agree_bit_for_bit(T, window, fmt, qk_norm):
    """A small grid takes 64 queries per workgroup, a large one (or one with moments) 128: the first member's rows and
    c_proj dots are the same bits alone, with moments, and among enough members to fill the GPU."""
    g = torch.Generator(DEV).manual_seed(36)
    m = 1 + 8 * 1024 // (T // 128 * 8)
    log_case(f'attention 64 / 128 queries T={T} window={window} format={fmt} qk_norm={qk_norm}')
    x = torch.randn(m * T, 3, 8, 64, device=DEV, generator=g)
    if qk_norm:
        x[:, :2] *= torch.rsqrt(x[:, :2].square().mean(-1, keepdim=True))
    if fmt == _lib.QK_F16_Q_LOG2:
        x[:, 0] *= 0.18033688
    half = fmt in (_lib.QK_F16, _lib.QK_F16_Q_LOG2)
    rows = x.half().view(torch.bfloat16) if half else x.bfloat16()
    if fmt == _lib.QK_BF16:
        rows[:, 2] = rows[:, 2].half().view(torch.bfloat16)
    b = torch.randn(m, 512, device=DEV, generator=g)

    def run(members, moments):
        y = torch.empty(members * T, 512, device=DEV, dtype=torch.bfloat16)
        u, mom = torch.empty(members * T, 8, device=DEV), torch.empty(members, 8, 2, 64, device=DEV)
        n = _lib.size_query('noise_attention_workspace_size', members, T)
        ws = torch.empty(n, device=DEV, dtype=torch.uint8)
        _lib.call('noise_attention', rows.data_ptr(), members, T, window, qk_norm, fmt, b.data_ptr(), 0, y.data_ptr(),
                  u.data_ptr(), mom.data_ptr() if moments else None, ws.data_ptr() if moments else None,
                  n if moments else 0, _stream())
        torch.cuda.synchronize()
        return y[:T], u[:T]
    alone = run(1, False)
    for other in (run(1, True), run(m, False)):
        assert torch.equal(alone[0], other[0]) and torch.equal(alone[1], other[1])
    # (the same kernel's numbers against the oracle: test_attention_matches_oracle_and_moments)
    assert torch.isfinite(alone[0].float()).all()


def test_adam_of_whole_and_ragged_blocks_at_any_address():
    """Tensors of whole and ragged blocks, at 16-byte addresses and one element off: the same bits, and nothing written
    past the end."""
    import math
    g = torch.Generator().manual_seed(37)
    for n in (1, 255, 257, 511, 513, 2047, 2048, 2049, 3 * 2048 + 1023):
        log_case(f'adam n={n}')
        vals = [torch.randn(n, generator=g), torch.randn(n, generator=g), torch.randn(n, generator=g),
                torch.rand(n, generator=g)]
        res = []
        for off in (0, 1):
            bufs = [torch.full((n + 9,), 7.0, device=DEV) for _ in vals]
            for buf, v in zip(bufs, vals):
                buf[off:off + n] = v.to(DEV)
            p, gr, m, v = (buf[off:off + n] for buf in bufs)
            _lib.call('noise_adam', p.data_ptr(), gr.data_ptr(), m.data_ptr(), v.data_ptr(), n, 1e-3, 0.5, 0.95, 1e-8,
                      math.sqrt(1 - 0.95), _stream())
            torch.cuda.synchronize()
            assert all((buf[off + n:] == 7).all() and (buf[:off] == 7).all() for buf in bufs)
            res.append((p.clone(), m.clone(), v.clone()))
        for x, y in zip(*res):
            assert torch.equal(x, y)


@pytest.mark.parametrize('count', [1, 2, 64, 65, 129])
def test_adam_batch_is_each_tensor_alone(count):
    """Batches of one tensor, of several, of as many as one launch takes and of more: every tensor gets the bits of a call
    of its own, with its own step size, and no other element of the flat buffers changes."""
    g = torch.Generator().manual_seed(47)
    log_case(f'adam batch of {count}')
    sizes = [(1, 511, 256, 513, 1000, 512)[k % 6] for k in range(count)]
    total = sum(sizes) + 3 * count
    start = [torch.randn(total, generator=g) for _ in range(3)] + [torch.rand(total, generator=g)]
    batch, single = ([t.to(DEV) for t in start] for _ in range(2))

    def items(bufs):
        at, out = 0, []
        for k, n in enumerate(sizes):
            out.append((*(t.data_ptr() + 4 * at for t in bufs), n, 1e-3 / (k + 1), 0.2 + 0.001 * k))
            at += n + 3
        return out
    ptr, c, _keep = _lib.adam_tensors(items(batch))
    _lib.call('noise_adam_batch', ptr, c, 0.5, 0.95, 1e-8, _stream())
    for p, gr, m, v, n, step, bc2 in items(single):
        _lib.call('noise_adam', p, gr, m, v, n, step, 0.5, 0.95, 1e-8, bc2, _stream())
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(batch, single))
    at = 0
    for n in sizes:
        for t, before in zip(batch, start):
            assert torch.equal(t[at + n:at + n + 3].cpu(), before[at + n:at + n + 3])
        at += n + 3


@pytest.mark.parametrize('pairs', [2, 15, 16, 17, 2047, 2049])
def test_rank_fitness_of_small_populations_with_ties(pairs):
    """Sixteen threads per pair, around whole workgroups of 16 pairs and whole tiles of 2048: the oracle's centred ranks
    bit for bit, many of them ties."""
    from oracle import eggroll as oe
    g = torch.Generator().manual_seed(38)
    log_case(f'rank fitness pairs={pairs}')
    losses = 8 + torch.randint(0, 50, (2 * pairs,), generator=g) / 64
    fit, weight = torch.empty(pairs, device=DEV), torch.empty(pairs, device=DEV)
    dl = losses.to(DEV)
    _lib.call('noise_fitness', dl.data_ptr(), 2 * pairs, pairs, _lib.FITNESS_RANK, fit.data_ptr(), weight.data_ptr(),
              _stream())
    torch.cuda.synchronize()
    ref, _ = oe.rank_fitness(losses, pairs)
    assert torch.equal(fit.cpu(), ref)


@pytest.mark.parametrize('off', [0, 1])
def test_batched_weight_casts_equal_the_single_ones(off):
    """noise_cast_weights over more matrices than one launch holds, ragged sizes, both layouts, aligned and misaligned
    sources: noise_cast_bf16 and noise_weight_tiles bit for bit, and nothing written past a matrix."""
    g = torch.Generator().manual_seed(39)
    shapes = [(64, 32), (512, 2048), (1, 1), (3, 7), (5, 4096), (1, 4097), (128, 96)] + [(2, 9)] * 63
    log_case(f'batched weight casts, source offset {off}')
    src = [torch.randn(r * c + 1, generator=g).to(DEV)[off:off + r * c] for r, c in shapes]
    tiled = [r % 64 == 0 and c % 32 == 0 for r, c in shapes]
    out = [torch.full((r * c + 8,), 7., device=DEV, dtype=torch.bfloat16) for r, c in shapes]
    ptr, n, _keep = _lib.casts([(x.data_ptr(), o.data_ptr(), r, c, _lib.LAYOUT_WTILE if t else _lib.LAYOUT_ROWS)
                                for x, o, (r, c), t in zip(src, out, shapes, tiled)])
    _lib.call('noise_cast_weights', ptr, n, _stream())
    for x, o, (r, c), t in zip(src, out, shapes, tiled):
        ref = torch.empty(r * c, device=DEV, dtype=torch.bfloat16)
        _lib.call('noise_cast_bf16', x.data_ptr(), ref.data_ptr(), r * c, 0, _stream())
        if t:
            rows, ref = ref, torch.empty_like(ref)
            _lib.call('noise_weight_tiles', rows.data_ptr(), r, c, ref.data_ptr(), _stream())
        torch.cuda.synchronize()
        assert torch.equal(o[:r * c], ref) and (o[r * c:] == 7).all(), (r, c)


@pytest.mark.parametrize('na,nb', [(1, 0), (5, 300), (8192, 8192), (8193, 1), (100003, 7)])
def test_token_range(na, nb):
    """The id check's partials over fewer ids than one workgroup, exactly the launch, and past it: the exact extremes."""
    from noise_amd.population import token_range
    g = torch.Generator().manual_seed(40)
    log_case(f'token_range {na} {nb}')
    a = torch.randint(-2 ** 62, 2 ** 62, (na,), generator=g)
    b = torch.randint(-2 ** 62, 2 ** 62, (nb,), generator=g) if nb else None
    want = (int(a.min()), int(a.max())) + ((int(b.min()), int(b.max())) if nb else ())
    assert token_range(a.to(DEV), None if b is None else b.to(DEV))() == want


def test_forward_stage_by_stage_equals_the_whole_pass():
    """noise_forward one stage at a time (as a stage timer drives it), in chunks whose noise rows start past 0, and in one
    call: the same losses bit for bit."""
    from noise_amd import population
    from noise_amd.model import make_model
    from noise_amd.synthetic import antithetic_signs, population_noise, trained_like, zipf_tokens
    m, T = 6, 128
    log_case('forward stage by stage')
    model = trained_like(make_model('cpu', 0)).to(DEV)
    p = dict(model.named_parameters())
    noise = {n: tuple(t.to(DEV) for t in v) if isinstance(v, tuple) else v.to(DEV)
             for n, v in population_noise({n: tuple(t.shape) for n, t in p.items()}, m // 2, per_member=False).items()}
    idx, tgt = (t.to(DEV) for t in zipf_tokens(T))
    sign = antithetic_signs(m, 1e-2).to(DEV)

    def loss(chunk):
        return population.Population(model, chunk=chunk).loss(p, noise, sign, idx, tgt, pair_shift=1)
    whole = loss(m)
    assert torch.equal(loss(2), whole) and torch.equal(loss(4), whole)
    population.TIMER = timer = population.StageTimer()
    try:
        assert torch.equal(loss(m), whole)
    finally:
        population.TIMER = population._NoTimer()
    timer.collect()
    assert timer.count == {**{s: 8 for s in population.BLOCK_STAGES}, 'head': 1}


def _outer_case(g, shapes, n):
    mats = []
    for o, i, pad in shapes:
        a = torch.randn(n, o + pad, generator=g)[:, :o] if o else None
        mats.append((a, torch.randn(n, i + pad, generator=g)[:, :i]))
    return mats, torch.randn(n, generator=g)


def _outer_gpu(mats, w, scale):
    dev = [(None if a is None else _strided(a), _strided(b)) for a, b in mats]
    grads = [torch.full((max(1, 0 if a is None else a.shape[1]) * b.shape[1] + 4,), 7., device=DEV) for a, b in mats]
    wd = w.to(DEV)
    ptr, cnt, _keep = _lib.outer_mats([(0 if a is None else a.data_ptr(), 0 if a is None else a.stride(0), b.data_ptr(),
                                        b.stride(0), 1 if a is None else a.shape[1], b.shape[1], gr.data_ptr())
                                       for (a, b), gr in zip(dev, grads)])
    _lib.call('noise_outer_update_batch', ptr, cnt, wd.data_ptr(), len(w), scale, _stream())
    torch.cuda.synchronize()
    out = []
    for (a, b), gr in zip(mats, grads):
        assert (gr[-4:] == 7).all()  # nothing past the matrix
        out.append(gr[:-4].view(-1, b.shape[1]).cpu())
    return out


def _strided(t):
    """t on the GPU with the row stride it has on the host."""
    buf = torch.zeros(t.shape[0], t.stride(0), device=DEV)
    buf[:, :t.shape[1]] = t.to(DEV)
    return buf[:, :t.shape[1]]


@pytest.mark.parametrize('n', [1, 31, 33, 100])
def test_outer_update_of_ragged_matrices(n):
    """A matrix of more tiles than the GPU holds at once beside small ones, ragged outputs, padded and odd row strides, a
    vector parameter, direction counts around the 32-direction chunks: against the fp64 sum. w a is rounded once and an
    output adds n exact products in fp32, each addition rounding at most 2^-24 of what the magnitudes add up to (the
    scale is a power of two)."""
    g = torch.Generator().manual_seed(41)
    log_case(f'outer update, ragged matrices, {n} directions')
    mats, w = _outer_case(g, [(4100, 1000, 0), (130, 257, 3), (0, 8, 0), (8, 32, 1), (1, 1, 0), (128, 128, 4)], n)
    for (a, b), got in zip(mats, _outer_gpu(mats, w, -0.25)):
        wa = (torch.ones(n, 1) if a is None else a).double() * w.double()[:, None]
        ref, mag = wa.t() @ b.double() * -0.25, wa.abs().t() @ b.double().abs() * 0.25
        assert ((got.double() - ref).abs() <= (n + 2) * 2 ** -24 * mag).all()


def test_outer_update_is_the_same_bits_alone_and_in_a_batch():
    """A matrix's gradient depends neither on the matrices that share its launch nor on its position: 70 matrices, more
    than one launch takes, with far more tiles than the GPU holds at once, against a call for each."""
    g = torch.Generator().manual_seed(44)
    n = 75
    log_case('outer update, batch against single calls')
    shapes = [(4100, 1000, 0), (512, 512, 0), (70, 130, 1), (0, 8, 0)] + [(64 + 7 * k, 96 + 3 * k, k % 4) for k in range(66)]
    mats, w = _outer_case(g, shapes, n)
    batch = _outer_gpu(mats, w, -0.3)
    for k in (0, 1, 2, 3, 40, 63, 64, 69):
        assert torch.equal(_outer_gpu(mats[k:k + 1], w, -0.3)[0], batch[k]), shapes[k]


@pytest.mark.parametrize('scale_a', [2. ** -118, 2. ** 100])
def test_outer_update_keeps_24_bits_of_operands_of_any_size(scale_a):
    """Operands far from 1 have the same relative error as N(0, 1) ones, in an update of many tiles: the bound of
    test_outer_update_of_ragged_matrices (every product and sum stays a normal fp32 number)."""
    g = torch.Generator().manual_seed(45)
    n = 40
    log_case(f'outer update, operands of size {scale_a}')
    mats, w = _outer_case(g, [(4100, 1000, 0)], n)
    a, b = mats[0]
    a, b = a.sign() * (0.5 + torch.rand(a.shape, generator=g)) * scale_a, b.sign() * (0.5 + torch.rand(b.shape, generator=g))
    w = 0.5 + torch.rand(n, generator=g)
    got = _outer_gpu([(a, b)], w, 1.0)[0]
    wa = a.double() * w.double()[:, None]
    ref, mag = wa.t() @ b.double(), wa.abs().t() @ b.double().abs()
    assert ((got.double() - ref).abs() <= (n + 2) * 2 ** -24 * mag).all()


def test_outer_update_of_nan_weights():
    """z-score fitness of a population with one NaN loss makes every weight NaN: every gradient is NaN."""
    g = torch.Generator().manual_seed(46)
    log_case('outer update, NaN weights')
    mats, w = _outer_case(g, [(4100, 1000, 0), (0, 8, 0), (70, 130, 1)], 64)
    for got in _outer_gpu(mats, torch.full_like(w, float('nan')), -0.25):
        assert torch.isnan(got).all()


@pytest.mark.parametrize('pad,off', [(0, 1), (2, 0), (4, 3)])
def test_outer_update_of_rows_off_16_byte_addresses(pad, off):
    """Full tiles whose rows start off 16-byte addresses (by the pointer, the row stride or both): the bits of
    the aligned rows."""
    g = torch.Generator().manual_seed(43)
    log_case(f'outer update, row padding {pad}, offset {off}')
    n, o, i = 37, 4096, 1024
    a, b, w = (torch.randn(n, k, generator=g).to(DEV) for k in (o, i, 1))
    got = []
    for p, f in ((0, 0), (pad, off)):
        rows = []
        for t in (a, b):
            flat = torch.zeros(n * (t.shape[1] + p) + f, device=DEV)
            rows.append(flat[f:].view(n, -1)[:, :t.shape[1]])
            rows[-1].copy_(t)
        grad = torch.zeros(o, i, device=DEV)
        ptr, cnt, _keep = _lib.outer_mats([(rows[0].data_ptr(), o + p, rows[1].data_ptr(), i + p, o, i, grad.data_ptr())])
        _lib.call('noise_outer_update_batch', ptr, cnt, w.data_ptr(), n, 1.0, _stream())
        got.append(grad)
    torch.cuda.synchronize()
    assert torch.equal(got[0], got[1])
    ref = (a * w).double().cpu().t() @ b.double().cpu()
    assert (got[0].cpu().double() - ref).norm() <= 1e-6 * ref.norm()


def test_outer_update_of_non_finite_and_extreme_values():
    """Infinities, NaN and values near fp32's largest: what the fp32 sum gives, in that column or row only; tiny values (a
    product of 1e-30) keep their sum."""
    g = torch.Generator().manual_seed(42)
    n = 40
    log_case('outer update of non-finite and extreme values')
    mats, w = _outer_case(g, [(4100, 1000, 0)], n)
    a, b = mats[0]
    w = w.abs() + 0.5
    w[3] = 1
    b[3] = b[3].abs() + 0.1  # (no infinity times zero, and infinities of one sign per row)
    a[3, 5], a[3, 6], a[7, 2000], b[9, 700] = float('inf'), float('-inf'), float('nan'), float('inf')
    a[9] = a[9].abs() + 0.1
    a[:, 17], a[3, 17] = 0, 3.4e38  # with b[3, 1] = 2^-100 finite
    b[3, 1] = 2 ** -100
    a[:, 4000] *= 1e-30
    got = _outer_gpu(mats, w, 1.0)[0]
    ref = torch.zeros(4100, 1000)
    for j in range(n):
        ref += (w[j] * a[j])[:, None] * b[j][None]
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], ref[inf])
    ok = torch.isfinite(ref)
    mag = (w[:, None].double() * a.double()).abs().nan_to_num(0, 0, 0).t() @ b.double().abs().nan_to_num(0, 0, 0)
    assert ((got.double() - ref.double()).abs()[ok] <= ((4 + 6 * 2 + n) * 2 ** -23 * mag)[ok]).all()
    assert (got[4000, :700] != 0).all()


@pytest.mark.parametrize('members,T', [(1, 5), (3, 16), (2, 4096), (1, 8230), (5, 130)])
def test_loss_reductions_add_the_row_losses_in_their_fixed_order(members, T):
    """Member means, sum and mean of the head's losses, rows below one chain step, around whole LDS tiles of 4096 and past
    them, some targets ignored: bit for bit the sixteen strided fp32 chains of the per-row losses, added in order."""
    g = torch.Generator().manual_seed(43)
    V, M = 256, members * T
    log_case(f'loss reductions members={members} T={T}')
    x, w = torch.randn(M, 512, generator=g).to(DEV), (torch.randn(V, 512, generator=g) * 0.05).to(DEV)
    a, b, sign = torch.zeros(members, V, device=DEV), torch.zeros(members, 512, device=DEV), torch.zeros(members, device=DEV)
    tgt = torch.randint(0, V, (M,), generator=g)
    n = _lib.size_query('noise_head_ce_workspace_size', members, T, V, _lib.HEAD_FP32)
    ws = torch.empty(n, device=DEV, dtype=torch.uint8)

    def run(red, targets, size):
        t, loss = targets.to(DEV), torch.empty(size, device=DEV)
        _lib.call('noise_head_ce', x.data_ptr(), 0, None, w.data_ptr(), V, _lib.HEAD_FP32, a.data_ptr(), b.data_ptr(),
                  sign.data_ptr(), t.data_ptr(), T, members, T, 0, red, loss.data_ptr(), None, ws.data_ptr(), n, None, 0,
                  _stream())
        torch.cuda.synchronize()
        return loss.cpu()

    def chains(rows, valid):
        acc = torch.zeros(16)
        for i in range(0, len(rows), 16):
            k = min(16, len(rows) - i)
            acc[:k] = torch.where(valid[i:i + k], acc[:k] + rows[i:i + k], acc[:k])
        t = torch.zeros(())
        for v in acc:
            t = t + v
        return t
    rows = run(_lib.CE_NONE, tgt, M)
    every = torch.ones(T, dtype=torch.bool)
    means = torch.stack([chains(rows[p * T:(p + 1) * T], every) / torch.tensor(float(T)) for p in range(members)])
    assert torch.equal(run(_lib.CE_MEMBER_MEAN, tgt, members), means)
    tgt[::3] = -1
    valid, rows = tgt != -1, run(_lib.CE_NONE, tgt, M)
    total = chains(rows, valid)
    assert torch.equal(run(_lib.CE_SUM, tgt, 1)[0], total)
    assert torch.equal(run(_lib.CE_MEAN, tgt, 1)[0], total / valid.sum().float())
    if M > 16:
        assert torch.isnan(run(_lib.CE_MEAN, torch.full((M,), -1), 1)).all()


@pytest.mark.parametrize('kind', ['q', 'k'])
@pytest.mark.parametrize('n,b,T,window', [(3, 2, 128, 40), (70, 1, 256, 300), (9, 2, 1152, 1100)])
def test_scores_of_a_credit_chunk_equal_those_of_its_outputs(kind, n, b, T, window):
    """The attention epilogue's head scores (outputs never written) against noise_head_scores on the outputs of the same
    reruns, with fp32 and bf16, strided and misaligned baselines: the same 64 fp32 products added in another order, 64
    2^-23 of their magnitudes. Small grids (64 queries per workgroup) and ones that fill the GPU."""
    from noise_amd import credit
    g = torch.Generator(DEV).manual_seed(45)
    log_case(f'scores of a credit chunk {kind} n={n} b={b} T={T}')

    def heads(*shape):
        return torch.randn(*shape, T, 8, 64, device=DEV, generator=g)
    raw, a, fixed, values, target = heads(b), heads(n, b).bfloat16(), heads(b).bfloat16(), heads(b).bfloat16(), heads(b)
    cos, sin = torch.randn(T, 32, device=DEV, generator=g), torch.randn(T, 32, device=DEV, generator=g)
    args = (kind, raw, a, 0.5, cos, sin, fixed, values, window)
    out = credit.rerun(*args)
    base = heads(b)
    for base in (base, base.bfloat16(), base.transpose(1, 2).contiguous().transpose(1, 2),
                 torch.cat([base.new_zeros(1), base.flatten()])[1:].view(base.shape)):
        ref = credit.head_scores(out, base, target)
        got = credit.rerun_scores(*args, base, target)
        change = (out.double() - base.double()) * target.double()
        bound = 64 * 2 ** -23 * change.abs().sum(-1).permute(1, 3, 2, 0) + 1e-30
        assert got.shape == ref.shape and ((got.double() - ref.double()).abs() <= bound).all()


@pytest.mark.parametrize('members,T,pair', [(1, 1, 0), (2, 7, 1), (5, 33, 1), (9, 130, 0), (18, 4, 1)])
@pytest.mark.parametrize('din', [64, 512, 1088])
def test_linear_on_shared_activations_equals_separate_copies(members, T, pair, din):
    """The input-side dots take four rows (deeper than 512 columns: one) against one direction, or four against four where
    members share one activation: the same bits, for ragged row and direction groups, odd member counts and pairs."""
    from noise_amd import ops
    g = torch.Generator(DEV).manual_seed(46)
    log_case(f'linear on shared activations members={members} T={T} pair={pair} din={din}')
    dirs = (members + pair) >> pair
    x = torch.randn(T, din, device=DEV, generator=g).bfloat16()
    w = (torch.randn(128, din, device=DEV, generator=g) * din ** -0.5).bfloat16()
    a, b = torch.randn(dirs, 128, device=DEV, generator=g), torch.randn(dirs, din, device=DEV, generator=g)
    sign = torch.randn(members, device=DEV, generator=g)
    one = ops.lowrank_linear(x, w, a, b, sign, T=T, pair_shift=pair)
    own = ops.lowrank_linear(x[None].repeat(members, 1, 1).contiguous(), w, a, b, sign, T=T, pair_shift=pair)
    assert torch.equal(one, own)
    xd, wd, s = x.double(), w.double(), sign.double()[:, None, None]
    pick = torch.arange(members, device=DEV) >> pair
    av, bv = a.double()[pick][:, None], b.bfloat16().double()[pick]
    dense, u = xd @ wd.t(), (xd @ bv.t()).t()[..., None]
    ref = dense + s * u * av
    # the dense product and the dot are each rounded to bf16 (2^-8) after din fp32 additions
    mag = xd.abs() @ wd.abs().t() + s.abs() * (xd.abs() @ bv.abs().t()).t()[..., None] * av.abs()
    bound = 1.01 * 2 ** -8 * (dense.abs() + (s * u * av).abs()) + (din + 4) * 2 ** -23 * mag
    assert ((one.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize('first', [False, True])
@pytest.mark.parametrize('T', [136, 1096])
def test_block_entry_of_few_and_many_rows_agree_bit_for_bit(T, first):
    """Past 32 rows per CU (16 for blocks after the first and short members) the block entry runs workgroups of 8 rows,
    below it a wave per row: every member's stream, operand, dots and gates are the same bits in a launch of more than
    16,000 rows, in one of up to 6,000 and in one of its own."""
    g = torch.Generator(DEV).manual_seed(48)
    m, D, V = 16384 // T + 2, 512, 640
    M = m * T
    log_case(f'block entry of few and many rows T={T} first={first}')

    def rnd(*shape):
        return torch.randn(*shape, device=DEV, generator=g)
    x, y1, y2, u1, u2 = rnd(M, D), rnd(M, D).bfloat16(), rnd(M, D).bfloat16(), rnd(M, 8), rnd(M, 8)
    v = {k: rnd(m, n) for k, n in dict(a1=D, a2=D, er=1, e0=1, bq=D, bk=D, bv=D, ga=8, gb=32, ea=V, eb=D).items()}
    gw, w, lr, l0, sign = rnd(8, 32), rnd(V, D), rnd(1), rnd(1), 0.1 * rnd(m)
    idx = torch.randint(0, V, (T,), device=DEV, generator=g)

    def run(lo, hi):
        n, r = (hi - lo) * T, slice(lo * T, hi * T)
        xo, h = torch.empty(n, D, device=DEV), torch.empty(n, D, device=DEV, dtype=torch.bfloat16)
        u, gate = torch.empty(n, 4, device=DEV), torch.empty(n, 8, device=DEV)
        d = {k: t[lo:].data_ptr() for k, t in v.items()}
        pend, npend = _lib.pending((y1[r].data_ptr(), u1[r].data_ptr(), 8, 8, 1, d['a1']),
                                   (y2[r].data_ptr(), u2[r].data_ptr(), 8, 8, 1, d['a2']))
        _emb, emb = _lib.embed(w.data_ptr(), V, d['ea'], d['eb'], idx.data_ptr(), 0)
        _lib.call('noise_block_entry', None if first else x[r].data_ptr(), None, xo.data_ptr(), h.data_ptr(),
                  u.data_ptr(), d['bq'], d['bk'], d['bv'], lr.data_ptr(), l0.data_ptr(), d['er'], d['e0'], 1,
                  gw.data_ptr(), d['ga'], d['gb'], gate.data_ptr(), sign[lo:].data_ptr(), hi - lo, T, 0,
                  None if first else pend, 0 if first else npend, emb, _stream())
        torch.cuda.synchronize()
        return xo, h, u, gate
    whole = run(0, m)
    for lo, hi in ((0, 1), (m // 2, m // 2 + 1), (m - 1, m), (0, 6000 // T)):
        for some, all_ in zip(run(lo, hi), whole):
            assert torch.equal(some, all_[lo * T:hi * T])


@pytest.mark.parametrize('T', [128, 1152, 2048])
def test_moment_partials_around_eight(T):
    """1, 9 and 16 partials per head: the moments are the fixed-order fp32 sums of y and y^2 per 128 queries, within fp32
    rounding of fp64 means of the kernel's own output."""
    g = torch.Generator(DEV).manual_seed(47)
    log_case(f'moments T={T}')
    x = torch.randn(T, 3, 512, device=DEV, generator=g).bfloat16()
    x[:, 2] = x[:, 2].half().view(torch.bfloat16)
    y, mom = torch.empty(T, 512, device=DEV, dtype=torch.bfloat16), torch.empty(1, 8, 2, 64, device=DEV)
    n = _lib.size_query('noise_attention_workspace_size', 1, T)
    ws = torch.empty(n, device=DEV, dtype=torch.uint8)
    _lib.call('noise_attention', x.data_ptr(), 1, T, T, 0, _lib.QK_BF16, None, 0, y.data_ptr(), None, mom.data_ptr(),
              ws.data_ptr(), n, _stream())
    torch.cuda.synchronize()
    yd = y.double().view(T, 8, 64)
    ref, mag = torch.stack([yd.mean(0), yd.square().mean(0)], 1), torch.stack([yd.abs().mean(0), yd.square().mean(0)], 1)
    assert ((mom[0].double() - ref).abs() <= (T // 128 + 12) * 2 ** -23 * mag).all()


@pytest.mark.parametrize('members,T', [(1, 1), (3, 5), (2, 1501), (9, 333), (1, 2049)])
def test_head_of_ragged_rows_from_tiled_and_row_major_operands(members, T):
    """From 2048 rows on the fp32 head pads its tiled operand to whole 16-row groups; with a workspace that has no room for
    the padding it takes row-major operands. The losses are the same bits, and a workspace smaller still is refused."""
    g = torch.Generator(DEV).manual_seed(49)
    V, M = 512, members * T
    log_case(f'ragged fp32 head members={members} T={T}')
    x, w = torch.randn(M, 512, device=DEV, generator=g), torch.randn(V, 512, device=DEV, generator=g) * 0.05
    a, b = torch.randn(members, V, device=DEV, generator=g), torch.randn(members, 512, device=DEV, generator=g)
    sign = 0.01 * torch.randn(members, device=DEV, generator=g)
    tgt = torch.randint(0, V, (T,), device=DEV, generator=g)
    full = _lib.size_query('noise_head_ce_workspace_size', members, T, V, _lib.HEAD_FP32)
    least = full - (-M) % 16 * 1024
    assert least < full
    ws = torch.empty(full, device=DEV, dtype=torch.uint8)

    def run(size):
        loss = torch.full((M + 16,), 7., device=DEV)
        _lib.call('noise_head_ce', x.data_ptr(), 0, None, w.data_ptr(), V, _lib.HEAD_FP32, a.data_ptr(), b.data_ptr(),
                  sign.data_ptr(), tgt.data_ptr(), 0, members, T, 0, _lib.CE_NONE, loss.data_ptr(), None, ws.data_ptr(),
                  size, None, 0, _stream())
        torch.cuda.synchronize()
        assert (loss[M:] == 7).all()
        return loss[:M]
    tiled = run(full)
    assert torch.equal(tiled, run(least)) and torch.isfinite(tiled).all()
    with pytest.raises(_lib.NoiseHipError, match='NOISE_ENOSPC'):
        run(least - 1)
