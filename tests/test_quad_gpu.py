"""The four-wave tile kernel (csrc/quad_kernel.hpp) where it can go wrong: K of one stage, of an odd and an
even number of stages and ending inside one; rows and columns one past and one short of a tile, a half tile and
a block; every operand layout; D rows that take the vector path, that need element stores and that accumulate;
K ranges summed by the second launch.  Against the CPU oracle (dequantise, fp32 matmul).  The bound on
calc_diff is the repository's 1e-5; every element is also held to 1e-3 of itself or the root mean square (the
alignment of e4m3 products inside one MFMA leaves up to 1.4e-4 of it), plus one unit of a bf16 result."""
import ctypes
import threading

import pytest
import torch

import deep_gemm
from deep_gemm import _lib
from oracle import gemm as og, layout as ol
from helpers import gen, operand, calc_diff

pytestmark = pytest.mark.gpu
THRESH = 1e-5
TILES = ['256x256', '256x224', '256x160', '256x128', '128x128']


@pytest.fixture
def force(monkeypatch):
    def _set(tile, split=None):
        monkeypatch.setenv('DG_FORCE_BLOCK', tile)
        if split:
            monkeypatch.setenv('DG_SPLIT_K', str(split))
    return _set


def _check(d, ref):
    """calc_diff, and every element within one bf16 unit (2^-7 of it at most, two roundings of nearly equal
    sums) plus 1e-3 of the larger of it and the root mean square."""
    unit = 2.0 ** -7 if d.dtype == torch.bfloat16 else 0.0
    d, ref = d.double().cpu(), ref.double()
    assert calc_diff(d, ref) < THRESH
    rms = ref.pow(2).mean().sqrt()
    off = (d - ref).abs() - unit * ref.abs()
    worst = float((off / torch.maximum(ref.abs(), rms)).max())
    print(f'  worst element: {worst:.2e}', flush=True)
    assert worst <= 1e-3


def _fp8(m, n, k, seed, b_kind='e4m3'):
    g = gen(seed)
    a, sfa, a_deq = operand(m, k, 'e4m3', (1, 32), g)
    b, sfb, b_deq = operand(n, k, b_kind, (1, 32), g)
    return (a.cuda(), sfa.cuda()), (b.cuda(), sfb.cuda()), a_deq, b_deq


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('m,n,k', [
    (1, 1, 32), (255, 33, 128), (256, 160, 160), (257, 224, 256), (129, 225, 384), (191, 159, 640),
    (300, 257, 416), (513, 480, 528), (64, 97, 1040), (400, 512, 2048)])
def test_quad_k_major(force, tile, m, n, k):
    print(f'quad {tile} fp8 m={m} n={n} k={k}', flush=True)
    force(tile)
    a, b, a_deq, b_deq = _fp8(m, n, k, 1)
    for dt in (torch.bfloat16, torch.float32):
        d = torch.full((m, n), float('nan'), dtype=dt, device='cuda')
        deep_gemm.fp8_gemm_nt(a, b, d)
        _check(d, og.gemm_nt(a_deq, b_deq, dt))


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('m,n,k', [(255, 225, 128), (257, 96, 352), (130, 500, 704)])
def test_quad_fp4(force, tile, m, n, k):
    print(f'quad {tile} fp8 x fp4 m={m} n={n} k={k}', flush=True)
    force(tile)
    a, b, a_deq, b_deq = _fp8(m, n, k, 2, 'e2m1')
    d = torch.full((m, n), float('nan'), dtype=torch.bfloat16, device='cuda')
    deep_gemm.fp8_fp4_gemm_nt(a, b, d)
    _check(d, og.gemm_nt(a_deq, b_deq))


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('form', ['nn', 'tn', 'tt'])
@pytest.mark.parametrize('m,n,k', [(256, 224, 128), (272, 240, 416), (144, 496, 1152)])
def test_quad_mn_major(force, tile, form, m, n, k):
    print(f'quad {tile} {form} m={m} n={n} k={k}', flush=True)
    force(tile)
    (a, sfa), (b, sfb), a_deq, b_deq = _fp8(m, n, k, 3)
    if form[0] == 't':
        a, sfa = a.t().contiguous(), sfa.t().contiguous()
    if form[1] == 'n':
        b, sfb = b.t().contiguous(), sfb.t().contiguous()
    d = torch.full((m, n), float('nan'), dtype=torch.float32, device='cuda')
    getattr(deep_gemm, 'fp8_gemm_' + form)((a, sfa), (b, sfb), d)
    _check(d, og.gemm_nt(a_deq, b_deq, torch.float32))


@pytest.mark.parametrize('tile', ['256x256', '256x128', '128x128'])
@pytest.mark.parametrize('form', ['nt', 'nn', 'tn', 'tt'])
@pytest.mark.parametrize('m,n,k', [(256, 256, 64), (264, 120, 200), (136, 392, 520)])
def test_quad_bf16(force, tile, form, m, n, k):
    print(f'quad {tile} bf16 {form} m={m} n={n} k={k}', flush=True)
    force(tile)
    g = gen(4)
    a = (torch.randn(m, k, generator=g) * 0.1).bfloat16()
    b = (torch.randn(n, k, generator=g) * 0.1).bfloat16()
    x = (a if form[0] == 'n' else a.t().contiguous()).cuda()
    y = (b if form[1] == 't' else b.t().contiguous()).cuda()
    d = torch.full((m, n), float('nan'), dtype=torch.float32, device='cuda')
    getattr(deep_gemm, 'bf16_gemm_' + form)(x, y, d)
    _check(d, og.gemm_nt(a.float(), b.float(), torch.float32))


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('dt', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('n', [224, 231])
def test_quad_accumulate_bias(force, tile, dt, n):
    """D += A . B^T and a bias row, on rows of whole quartets and on rows that need element stores."""
    m, k = 270, 384
    print(f'quad {tile} accumulate / bias {dt} n={n}', flush=True)
    force(tile)
    a, b, a_deq, b_deq = _fp8(m, n, k, 5)
    ref = og.gemm_nt(a_deq, b_deq, torch.float32)
    scale = float(ref.abs().mean())
    c = (torch.randn(m, n, generator=gen(6)) * scale).to(dt)
    d = c.clone().cuda()
    deep_gemm.fp8_gemm_nt(a, b, d, c=d)
    _check(d, (ref + c.float()).to(dt))
    bias = (torch.randn(1, n, generator=gen(7)) * scale).to(dt)
    d = torch.full((m, n), float('nan'), dtype=dt, device='cuda')
    deep_gemm.fp8_gemm_nt(a, b, d, c=bias.cuda())
    _check(d, (ref + bias.float()).to(dt))


@pytest.mark.parametrize('kind', ['e4m3', 'e2m1', 'bf16'])
@pytest.mark.parametrize('n', [4, 12, 36, 100, 164, 236, 241, 246, 270, 511])
def test_quad_cut_rows(force, kind, n):
    """Rows of aligned quartets that end inside a block of columns (and inside a quartet): each output mode gives the
    columns of the call whose rows are whole, bit for bit, and what lies past the row stays as it was."""
    m, k = 270, 384
    ldd, full = -(-n // 8) * 8 + 8, -(-n // 256) * 256
    a, b, a_deq, b_deq = _fp8(m, full, k, 27, 'e2m1' if kind == 'e2m1' else 'e4m3')
    ref = og.gemm_nt(a_deq, b_deq, torch.float32)
    scale = float(ref.abs().mean())
    fn = deep_gemm.fp8_gemm_nt if kind == 'e4m3' else deep_gemm.fp8_fp4_gemm_nt
    if kind == 'bf16':
        fn, a, b = deep_gemm.bf16_gemm_nt, a_deq.bfloat16().cuda(), (b_deq / scale).bfloat16().cuda()
        ref, scale = og.gemm_nt(a.float().cpu(), b.float().cpu(), torch.float32), 1.0
    cut = (lambda x: x[:n].contiguous()) if kind == 'bf16' else (lambda x: tuple(t[:n].contiguous() for t in x))
    bias = (torch.randn(1, full, generator=gen(28)) * scale).cuda()
    old = (torch.randn(m, full, generator=gen(29)) * scale).cuda()
    for tile in ['256x256', '256x128', '128x128'] + (['256x224', '256x160'] if kind != 'bf16' else []):
        force(tile)
        for dt in (torch.bfloat16, torch.float32):
            for mode in ['plain', 'bias', 'accumulate'] + (['stochastic'] if dt == torch.bfloat16 and kind != 'bf16' else []):
                print(f'quad cut rows {tile} {kind} n={n} {dt} {mode}', flush=True)
                whole = old.to(dt).clone()
                buf = torch.full((m, ldd), 7.0, dtype=dt, device='cuda')
                d = buf[:, :n]
                d.copy_(whole[:, :n])
                keys_w, keys_c = {}, {}
                if mode == 'bias':
                    keys_w, keys_c = dict(c=bias.to(dt)), dict(c=bias[:, :n].to(dt).contiguous())
                elif mode == 'accumulate':
                    keys_w, keys_c = dict(c=whole), dict(c=d)
                elif mode == 'stochastic':
                    keys_w = keys_c = dict(epilogue=deep_gemm.epilogue.BF16StochasticRounding())
                fn(a, b, whole, **keys_w)
                fn(a, cut(b), d, **keys_c)
                last = n // 4 * 4 if mode == 'stochastic' else n   # (columns past the row hash as zeros)
                assert torch.equal(d[:, :last], whole[:, :last])
                assert bool((buf[:, n:] == 7.0).all())
                want = ref + (bias.to(dt).float().cpu() if mode == 'bias' else old.to(dt).float().cpu() if mode == 'accumulate' else 0)
                if mode != 'stochastic':
                    _check(d, want[:, :n].to(dt))
                else:
                    unit = d.float().cpu().abs() * 2.0 ** -7 + 1e-3 * scale
                    assert bool(((d.float().cpu() - want[:, :n]).abs() <= unit).all())


@pytest.mark.parametrize('tile', ['256x256', '256x160', '128x128'])
@pytest.mark.parametrize('n', [200, 256])
def test_quad_m_indices_padding(force, tile, n):
    """Rows of an m_indices layout that lie past their group inside a tile are written as zeros, the others not."""
    sizes, alignment, k = [1, 255, 256, 300, 130, 17], 256, 416
    print(f'quad m_indices {tile} n={n}', flush=True)
    force(tile)
    total, ps = ol.psum_from_sizes(sizes, alignment)
    layout = ol.m_indices_from_psum(ps, alignment, total)
    g = gen(30)
    a, sfa, a_deq = operand(total, k, 'e4m3', (1, 32), g)
    b, sfb, b_deq = operand(n, k, 'e4m3', (1, 32), g, batch=len(sizes))
    d = torch.full((total, n), float('nan'), dtype=torch.bfloat16, device='cuda')
    deep_gemm.m_grouped_fp8_gemm_nt_contiguous((a.cuda(), sfa.cuda()), (b.cuda(), sfb.cuda()), d, layout.cuda(), use_psum_layout=False)
    out, ref = d.cpu(), og.m_grouped_contiguous(a_deq, b_deq, layout, False, alignment)
    live = layout >= 0
    _check(out[live], ref[live])
    assert torch.equal(out[~live], torch.zeros_like(out[~live]))


@pytest.mark.parametrize('tile,split', [('256x256', 2), ('256x256', 5), ('128x128', 3), ('128x128', 11)])
@pytest.mark.parametrize('m,n,k', [(300, 260, 1408), (130, 127, 2000)])
def test_quad_split(force, tile, split, m, n, k):
    """K ranges of one or several stages; the bf16 D is the rounding of the fp32 D."""
    print(f'quad {tile} split {split} m={m} n={n} k={k}', flush=True)
    force(tile, split)
    a, b, a_deq, b_deq = _fp8(m, n, k, 8)
    out = {}
    for dt in (torch.float32, torch.bfloat16):
        d = torch.full((m, n), float('nan'), dtype=dt, device='cuda')
        deep_gemm.fp8_gemm_nt(a, b, d)
        _check(d, og.gemm_nt(a_deq, b_deq, dt))
        out[dt] = d
    assert torch.equal(out[torch.bfloat16], out[torch.float32].bfloat16())


@pytest.mark.parametrize('tile', TILES)
@pytest.mark.parametrize('kind,form', [('e4m3', 'nt'), ('e4m3', 'tn'), ('e2m1', 'nt'), ('bf16', 'nt'), ('bf16', 'nn')])
def test_quad_split_forms(force, tile, kind, form):
    """Partials of every tile's layout (the uneven halves of 224 and 160 columns too), operand kind and major; plain,
    accumulated and with a bias row."""
    if kind == 'bf16' and tile in ('256x224', '256x160'):
        pytest.skip('bf16 runs these tiles on the eight-wave kernel, without K splits')
    m, n, k = 272, 240, 1168
    g = gen(31)
    a, sfa, a_deq = operand(m, k, 'e4m3', (1, 32), g)
    b, sfb, b_deq = operand(n, k, 'e4m3' if kind == 'bf16' else kind, (1, 32), g)
    scale = 1.0
    if kind == 'bf16':
        a_deq, b_deq = (x / x.abs().mean() for x in (a_deq, b_deq))
        a, b = a_deq.bfloat16(), b_deq.bfloat16()
        a_deq, b_deq = a.float(), b.float()
    if form[0] == 't':
        a, sfa = a.t().contiguous(), sfa.t().contiguous()
    if form[1] == 'n':
        b, sfb = b.t().contiguous(), sfb.t().contiguous()
    ref = og.gemm_nt(a_deq, b_deq, torch.float32)
    scale = float(ref.abs().mean())
    x, y = (a.cuda(), b.cuda()) if kind == 'bf16' else ((a.cuda(), sfa.cuda()), (b.cuda(), sfb.cuda()))
    fn = getattr(deep_gemm, {'e4m3': 'fp8_gemm_', 'e2m1': 'fp8_fp4_gemm_', 'bf16': 'bf16_gemm_'}[kind] + form)
    bias = torch.randn(1, n, generator=gen(32)) * scale
    old = torch.randn(m, n, generator=gen(33)) * scale
    for split in (2, 5):
        print(f'quad split {split} {tile} {kind} {form}', flush=True)
        force(tile, split)
        d = torch.full((m, n), float('nan'), device='cuda')
        fn(x, y, d)
        _check(d, ref)
        fn(x, y, d, c=bias.cuda())
        _check(d, ref + bias)
        d = old.clone().cuda()
        fn(x, y, d, c=d)
        _check(d, ref + old)


@pytest.mark.parametrize('tile', ['256x256', '256x160', '128x128'])
def test_quad_split_batched(force, tile):
    bsz, m, n, k = 3, 140, 264, 1056
    print(f'quad split bmm {tile}', flush=True)
    force(tile, 3)
    g = gen(34)
    a, sfa, a_deq = operand(m, k, 'e4m3', (1, 32), g, batch=bsz)
    b, sfb, b_deq = operand(n, k, 'e4m3', (1, 32), g, batch=bsz)
    d = torch.full((bsz, m, n), float('nan'), device='cuda')
    deep_gemm.fp8_bmm((a.cuda(), sfa.cuda()), (b.cuda(), sfb.cuda()), d)
    for i in range(bsz):
        _check(d[i], og.gemm_nt(a_deq[i], b_deq[i], torch.float32))


@pytest.mark.parametrize('b_kind', ['e4m3', 'e2m1'])
@pytest.mark.parametrize('n', [2080, 2076])
def test_quad_d_past_the_caches(b_kind, n):
    """A D of more than 192 MiB at short K is stored past the caches; with rows that end at, and inside, a block."""
    m, k = 49157, 160
    print(f'quad stores past the caches {b_kind} n={n}', flush=True)
    assert 2 * m * n >= 192 << 20
    a, b, a_deq, b_deq = _fp8(m, n, k, 35, b_kind)
    d = torch.full((m, n), float('nan'), dtype=torch.bfloat16, device='cuda')
    (deep_gemm.fp8_gemm_nt if b_kind == 'e4m3' else deep_gemm.fp8_fp4_gemm_nt)(a, b, d)
    _check(d, og.gemm_nt(a_deq, b_deq))


@pytest.mark.parametrize('b_kind', ['e4m3', 'e2m1'])
def test_quad_anchored_live_blocks(b_kind):
    """384-row tiles of an M-grouped layout, whose loop leaves out the dead blocks of the second 192 rows: groups
    that end one short of, at and one past each count of live blocks; the default plan of alignment 32."""
    sizes = [1, 31, 192, 193, 223, 224, 225, 256, 257, 288, 289, 320, 321, 352, 353, 383, 384, 385, 0, 577]
    alignment, n, k = 32, 200, 416
    print(f'quad anchored {b_kind} sizes={sizes}', flush=True)
    total, ps = ol.psum_from_sizes(sizes, alignment)
    g = gen(9)
    a, sfa, a_deq = operand(total, k, 'e4m3', (1, 32), g)
    b, sfb, b_deq = operand(n, k, b_kind, (1, 32), g, batch=len(sizes))
    layout = torch.tensor(ps, dtype=torch.int32)
    old = deep_gemm.get_mk_alignment_for_contiguous_layout()
    deep_gemm.set_mk_alignment_for_contiguous_layout(alignment)
    try:
        d = torch.full((total, n), float('nan'), dtype=torch.bfloat16, device='cuda')
        fn = deep_gemm.m_grouped_fp8_gemm_nt_contiguous if b_kind == 'e4m3' else deep_gemm.m_grouped_fp8_fp4_gemm_nt_contiguous
        fn((a.cuda(), sfa.cuda()), (b.cuda(), sfb.cuda()), d, layout.cuda())
    finally:
        deep_gemm.set_mk_alignment_for_contiguous_layout(old)
    out, ref = d.cpu(), og.m_grouped_contiguous(a_deq, b_deq, layout, True, alignment)
    end = 0
    for size, stop in zip(sizes, ps):
        start, end = end, -(-stop // alignment) * alignment
        assert stop == start + size
        if size:
            _check(out[start:stop], ref[start:stop])
        assert torch.equal(out[stop:end], torch.zeros_like(out[stop:end]))


@pytest.mark.parametrize('tile', ['256x256', '256x128', '128x128'])
def test_quad_masked_order(force, tile):
    """Several tile rows per group: every live tile is served once and dead rows stay as they were, for more
    groups than a wave has lanes, groups without rows and counts at the tiles' edges."""
    g_num, max_m, n, k = 70, 520, 264, 160
    print(f'quad masked {tile}', flush=True)
    force(tile)
    g = gen(10)
    masked = torch.randint(0, 40, (g_num,), generator=g, dtype=torch.int32)
    masked[:12] = torch.tensor([520, 0, 0, 1, 127, 128, 129, 256, 257, 384, 385, 512], dtype=torch.int32)
    masked[64:67] = torch.tensor([0, 300, 520], dtype=torch.int32)
    a, sfa, a_deq = operand(max_m, k, 'e4m3', (1, 32), g, batch=g_num)
    b, sfb, b_deq = operand(n, k, 'e4m3', (1, 32), g, batch=g_num)
    d = torch.full((g_num, max_m, n), float('nan'), dtype=torch.bfloat16, device='cuda')
    deep_gemm.m_grouped_fp8_gemm_nt_masked((a.cuda(), sfa.cuda()), (b.cuda(), sfb.cuda()), d, masked.cuda(), 64)
    out, ref = d.cpu(), og.m_grouped_masked(a_deq, b_deq, masked)
    for i in range(g_num):
        rows = int(masked[i])
        assert torch.isnan(out[i, rows:].float()).all(), i
        if rows:
            assert calc_diff(out[i, :rows], ref[i, :rows]) < THRESH, i


def _split_call(seed, m=300, n=2112, k=7168):
    """A call whose default plan splits K on the four-wave tiles, and its eager result."""
    plan = deep_gemm.launch_plan(m, n, k)
    assert plan['split_k'] > 1 and plan['block_m'] >= 128, plan
    a, b, a_deq, b_deq = _fp8(m, n, k, seed)
    a = (a[0], deep_gemm.transform_sf_into_required_layout(a[1], m, k, (1, 32), is_sfa=True))
    b = (b[0], deep_gemm.transform_sf_into_required_layout(b[1], n, k, (1, 32), is_sfa=False))
    d = torch.empty(m, n, dtype=torch.float32, device='cuda')
    deep_gemm.fp8_gemm_nt(a, b, d)
    _check(d, og.gemm_nt(a_deq, b_deq, torch.float32))
    return a, b, d.clone()


def test_quad_split_captured_unsplit():
    """A graph of a call that splits K when run eagerly, replayed beside eager calls of its capture stream: the
    graph holds one unsplit launch, so neither side touches the other's partials."""
    print('quad split captured', flush=True)
    (a, b, ref), (a2, b2, ref2) = _split_call(21), _split_call(22)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    d, d2 = torch.empty_like(ref), torch.empty_like(ref)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        deep_gemm.fp8_gemm_nt(a, b, d)       # the stream has its workspace before the capture
    s.synchronize()
    assert torch.equal(d, ref)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        deep_gemm.fp8_gemm_nt(a, b, d)
    for i in range(4):
        d.fill_(float(i + 1))
        torch.cuda.synchronize()
        with torch.cuda.stream(t):
            graph.replay()
        with torch.cuda.stream(s):
            deep_gemm.fp8_gemm_nt(a2, b2, d2)
        torch.cuda.synchronize()
        _check(d, ref.cpu())
        assert torch.equal(d2, ref2), i


def test_quad_split_two_threads_on_a_stream():
    """Two host threads on one stream: each call's two launches stay together."""
    print('quad split two threads', flush=True)
    calls = [_split_call(23), _split_call(24)]
    outs = [[torch.empty_like(calls[0][2]) for _ in range(20)] for _ in calls]
    torch.cuda.synchronize()
    start = threading.Barrier(2)

    def work(i):
        start.wait(timeout=30)
        for d in outs[i]:
            deep_gemm.fp8_gemm_nt(calls[i][0], calls[i][1], d)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join(timeout=60)
    torch.cuda.synchronize()
    for i in range(2):
        for d in outs[i]:
            assert torch.equal(d, calls[i][2])


def test_quad_split_per_thread_streams():
    """hipStreamPerThread names another stream in every thread: calls of two threads share no partials (they run
    unsplit)."""
    print('quad split per-thread streams', flush=True)
    lib = _lib.load()
    m, n, k = 300, 2112, 7168
    calls = []
    for seed in (25, 26):
        a, b, _ = _split_call(seed)
        args = _lib.GemmArgs()
        args.kind, args.gemm_type, args.m, args.n, args.k, args.num_groups = _lib.DG_KIND_FP8_FP8, _lib.DG_GEMM_NORMAL, m, n, k, 1
        args.a, args.b, args.sfa, args.sfb = a[0].data_ptr(), b[0].data_ptr(), a[1].data_ptr(), b[1].data_ptr()
        args.lda, args.ldb, args.ldd = k, k, n
        args.sfa_ld, args.sfb_ld = a[1].stride(-1), b[1].stride(-1)
        args.d_dtype, args.alpha, args.alignment, args.library_workspace, args.split_k = _lib.DG_DTYPE_F32, 1.0, 256, 1, 1
        ref = torch.empty(m, n, device='cuda')
        args.d = ref.data_ptr()
        _lib.check(lib.dg_gemm(ctypes.byref(args), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), lib)
        args.split_k = 0
        calls.append((args, (a, b), ref, [torch.empty_like(ref) for _ in range(20)]))
    torch.cuda.synchronize()
    start, codes = threading.Barrier(2), []

    def work(args, outs):
        start.wait(timeout=30)
        for d in outs:
            args.d = d.data_ptr()
            codes.append(lib.dg_gemm(ctypes.byref(args), ctypes.c_void_p(2)))
    threads = [threading.Thread(target=work, args=(c[0], c[3])) for c in calls]
    for th in threads:
        th.start()
    for th in threads:
        th.join(timeout=60)
    torch.cuda.synchronize()
    assert codes == [0] * 40
    for _, _, ref, outs in calls:
        assert all(torch.equal(d, ref) for d in outs)
