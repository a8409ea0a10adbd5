"""The many-row matmul (k_q4_gemm_w) against the few-row kernels, bit for bit: a row's sums depend on the row alone, so
M rows in one call equal the same rows in calls of 16 (which tests/test_gpu_q4.py and test_gpu_q8.py hold to the oracle).
Sizes at the edges of its tiles (32 rows, 64 with two row tiles a wavefront; 128 or 64 columns a workgroup), of its
launch choices and of the k-slices (short last slices, an odd number of slices taken two at a time), ragged N and K."""
import ctypes as C

import numpy as np
import pytest
import torch  # noqa: F401 (its HIP runtime is the process's: loaded before the library)

import sllm_next as S
from tests import gpu_util as U

pytestmark = pytest.mark.gpu
STORE, ADD, SWIGLU = 0, 1, 2


def weights(r, N, K, wt):
    f = S.quantize_q4_0 if wt == 2 else None
    x = (r.standard_normal((N, K)) * 0.02).astype(np.float32)
    if wt == 2:
        return f(x)
    out = np.empty(N * (K // 32) * 34, np.uint8)
    S.lib().snx_quantize_q8_0(S._p(x), S._p(out), x.size)
    return out


def matmul(L, wt, w, x, N, epi, ldy, y0, off=0):
    """y0 with the product of rows x written (or added) at element offset `off` of a larger buffer"""
    M, K = x.shape
    xa, y = U.empty(L.snk_xa_bytes(M, K)), U.dev(y0)
    assert L.snk_quant_act(U.ptr(U.dev(x)), M, K, K, None, 1e-6, U.ptr(xa), U.stream()) == 0
    nb = (L.snk_q4_workspace_bytes if wt == 2 else L.snk_q8_workspace_bytes)(M, N, K)
    ws = U.empty(nb)
    f = L.snk_q4_gemm if wt == 2 else L.snk_q8_gemm
    assert f(U.ptr(w), U.ptr(xa), M, N, K, C.c_void_p(y.data_ptr() + 4 * off), ldy, epi, U.ptr(ws), nb, U.stream()) == 0
    return U.host(y, np.float32, y0.shape)


CASES = [  # wt, M, N, K, epi, ldy - columns, offset of y in floats
    (2, 256, 1000, 4096, STORE, 0, 0),      # two slices at a time; ragged columns
    (2, 257, 2560, 1280, ADD, 3, 1),        # 3 slices of 4 groups, one row past the tiles, y unaligned
    (2, 333, 2576, 9728 // 2, STORE, 5, 0),  # a short last slice
    (2, 192, 6144, 2560, STORE, 0, 0),      # below 256 rows
    (2, 100, 19456, 1056, SWIGLU, 0, 0),    # wide at 100 rows; K not a multiple of 128
    (2, 384, 19456, 1024, SWIGLU, 0, 0),    # two row tiles a wavefront, one slice
    (2, 480, 19456, 1056, STORE, 0, 0),     # the same with an odd number of 32-row tiles: the last workgroup's upper
    (2, 465, 19456, 1056, SWIGLU, 0, 0),    # one is past the operand
    (2, 512, 12320, 2080, ADD, 0, 2),       # two row tiles, ragged columns and K, y off 16 bytes
    (2, 260, 1056, 2048, SWIGLU, 1, 0),     # F a multiple of 16 alone, rows of h unaligned
    (8, 256, 1040, 2560, STORE, 0, 0),      # Q8_0: two slices at a time
    (8, 300, 6160, 1280, ADD, 0, 0),        # Q8_0: one slice at a time
    (8, 200, 4096, 1024, SWIGLU, 4, 0),
]


@pytest.mark.parametrize("wt,M,N,K,epi,pad,off", CASES)
def test_many_rows_are_the_few_rows_bits(wt, M, N, K, epi, pad, off):
    L, r = S.lib(), np.random.default_rng(M * 7 + N)
    raw = U.dev(weights(r, N, K, wt))
    w = U.empty((L.snk_q4_stripes_bytes if wt == 2 else L.snk_q8_tiles_bytes)(N, K))
    assert (L.snk_q4_repack if wt == 2 else L.snk_q8_repack)(U.ptr(raw), N, K, U.ptr(w), U.stream()) == 0
    x = r.standard_normal((M, K)).astype(np.float32)
    cols = N // 2 if epi == SWIGLU else N
    ldy = cols + pad
    y0 = r.standard_normal(M * ldy + off + 8).astype(np.float32)
    want = y0.copy()
    for m in range(0, M, 16):
        n = min(16, M - m)
        part = want[off + m * ldy:off + m * ldy + n * ldy].copy()
        want[off + m * ldy:off + m * ldy + n * ldy] = matmul(L, wt, w, x[m:m + n], N, epi, ldy, part)
    got = matmul(L, wt, w, x, N, epi, ldy, y0, off)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def same(a, b):
    """Equal bits where finite, and not finite in the same places."""
    f = np.isfinite(a)
    return np.array_equal(f, np.isfinite(b)) and np.array_equal(a[f].view(np.uint32), b[f].view(np.uint32))


def odd_rows(r, M, K):
    """Rows of ordinary values, and in each 32-row tile some whose values leave the formats: an infinity, a NaN, a block
    whose fp16 scale overflows, one of subnormal scale, zeros."""
    x = r.standard_normal((M, K)).astype(np.float32)
    for m in range(0, M, 32):
        for i, v in enumerate((np.inf, -np.inf, np.nan, 1e9)):
            if m + 5 * i + 1 < M:
                x[m + 5 * i + 1, (37 * (m + i)) % K] = v
        x[m] *= 1e-6
        x[min(m + 2, M - 1)] = 0
    return x


@pytest.mark.parametrize("wt,M,N,K,epi", [
    (2, 256, 1008, 1152, STORE), (2, 300, 6144, 1280, ADD), (2, 480, 19456, 1056, STORE), (2, 256, 4096, 1152, SWIGLU),
    (8, 256, 1008, 1152, STORE), (8, 300, 6144, 1280, SWIGLU),
])
def test_infinities_and_nans_stay_in_their_rows(wt, M, N, K, epi):
    """Rows that hold infinities, NaN or overflowing scales are not finite where the few-row kernels' are not, and every
    other row keeps its bits."""
    L, r = S.lib(), np.random.default_rng(M + N)
    w = U.empty((L.snk_q4_stripes_bytes if wt == 2 else L.snk_q8_tiles_bytes)(N, K))
    assert (L.snk_q4_repack if wt == 2 else L.snk_q8_repack)(U.ptr(U.dev(weights(r, N, K, wt))), N, K, U.ptr(w), U.stream()) == 0
    x = odd_rows(r, M, K)
    cols = N // 2 if epi == SWIGLU else N
    y0 = r.standard_normal((M, cols)).astype(np.float32)
    got = matmul(L, wt, w, x, N, epi, cols, y0)
    for m in range(0, M, 16):
        want = matmul(L, wt, w, x[m:m + 16], N, epi, cols, y0[m:m + 16])
        assert same(got[m:m + 16], want), m


@pytest.mark.parametrize("M,K,norm", [(192, 2560, False), (640, 2560, True), (336, 5120, True)])
def test_operand_of_infinities_and_nans(M, K, norm):
    """The activation quantizer's tile form over such rows: the row kernel's operand, bit for bit (a NaN as a NaN)."""
    L, r = S.lib(), np.random.default_rng(M)
    x, nw = odd_rows(r, M, K), U.dev((1 + 0.1 * r.standard_normal(K)).astype(np.float32))

    def operand(rows):
        xa = U.empty(L.snk_xa_bytes(len(rows), K))
        assert L.snk_quant_act(U.ptr(U.dev(rows)), len(rows), K, K, U.ptr(nw) if norm else None, 1e-6, U.ptr(xa),
                               U.stream()) == 0
        rec = U.host(xa, np.uint8)[:L.snk_xa_bytes(len(rows), K)].reshape(-1, 4864)
        q = rec[:, :4096].copy().view(np.uint16)
        k = rec[:, 4096:].copy().view(np.uint32)
        q[np.isnan(q.view(np.float16))], k[np.isnan(k.view(np.float32))] = 0x7e00, 0x7fc00000
        return q, k

    q, k = operand(x)
    n = L.snk_xa_bytes(32, K) // 2 // 4864  # a row tile's records
    for m in range(0, M, 16):
        wq, wk = operand(x[m:m + 16])
        t = slice(m // 16 * n, (m // 16 + 1) * n)
        assert np.array_equal(q[t], wq[:n]) and np.array_equal(k[t], wk[:n]), m


@pytest.mark.parametrize("wt,N,K,M,many", [
    (2, 256, 4096, 255, False), (8, 256, 4096, 200, False),   # narrow and deep: few tiles, a long walk
    (2, 1024, 3072, 255, False), (2, 1024, 1536, 224, False), (8, 768, 3072, 240, False),
    (2, 1024, 2048, 207, False), (2, 1024, 2048, 208, True),  # the line
    (8, 1000, 2080, 201, False), (2, 1000, 2080, 202, True),  # a short last slice counts whole
    (2, 768, 1024, 191, False), (2, 768, 1024, 192, True), (2, 256, 4096, 256, True),
    (2, 2560, 4096, 192, True), (8, 6144, 2560, 200, True),
])
def test_below_256_rows_narrow_matrices_keep_their_split_launches(wt, N, K, M, many):
    """Which launches a matmul takes, seen in its workspace (the split launches leave their slice sums there, the
    many-row kernel nothing): narrow and deep matrices of 192 to 255 rows, whose few wide tiles would leave most of the
    chip idle through the whole walk, stay split. The rows are the few rows' bits either way."""
    L, r = S.lib(), np.random.default_rng(N + K + M)
    w = U.empty((L.snk_q4_stripes_bytes if wt == 2 else L.snk_q8_tiles_bytes)(N, K))
    assert (L.snk_q4_repack if wt == 2 else L.snk_q8_repack)(U.ptr(U.dev(weights(r, N, K, wt))), N, K, U.ptr(w), U.stream()) == 0
    x = r.standard_normal((M, K)).astype(np.float32)
    xa, y = U.empty(L.snk_xa_bytes(M, K)), U.empty(4 * M * N)
    assert L.snk_quant_act(U.ptr(U.dev(x)), M, K, K, None, 1e-6, U.ptr(xa), U.stream()) == 0
    nb = (L.snk_q4_workspace_bytes if wt == 2 else L.snk_q8_workspace_bytes)(M, N, K)
    ws = torch.full((nb,), 0xA5, dtype=torch.uint8, device="cuda")
    f = L.snk_q4_gemm if wt == 2 else L.snk_q8_gemm
    assert f(U.ptr(w), U.ptr(xa), M, N, K, U.ptr(y), N, STORE, U.ptr(ws), nb, U.stream()) == 0
    assert bool((ws == 0xA5).all()) == many
    got = U.host(y, np.float32, (M, N))
    want = matmul(L, wt, w, x[:16], N, STORE, N, np.zeros(16 * N + 8, np.float32))[:16 * N].reshape(16, N)
    assert np.array_equal(got[:16].view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("M,K,norm", [(160, 2016, False), (131, 2560, False), (489, 2560, True), (613, 2080, True), (33, 9728, False),
                                      (160, 2560, False), (199, 2016, False), (43, 9728, False), (625, 2560, True),
                                      (771, 2080, True), (520, 4096, True), (331, 5120, True)])
def test_operand_of_many_rows_is_the_row_kernels(M, K, norm):
    """The activation quantizer's tile form (ragged last tiles, K not a multiple of 128, with and without the norm)
    against calls of 16 rows: the same integers and scales."""
    L, r = S.lib(), np.random.default_rng(M + K)
    x = (r.standard_normal((M, K)) * np.exp(r.standard_normal((M, 1)))).astype(np.float32)
    nw = U.dev((1 + 0.1 * r.standard_normal(K)).astype(np.float32))

    def operand(rows):
        xa = U.empty(L.snk_xa_bytes(len(rows), K))
        assert L.snk_quant_act(U.ptr(U.dev(rows)), len(rows), K, K, U.ptr(nw) if norm else None, 1e-6, U.ptr(xa),
                               U.stream()) == 0
        return U.xa_decode(U.host(xa, np.uint8), len(rows), K)

    q, d = operand(x)
    for m in range(0, M, 16):
        wq, wd = operand(x[m:m + 16])
        assert np.array_equal(q[m:m + 16], wq) and np.array_equal(d[m:m + 16].view(np.uint32), wd.view(np.uint32))


def least_us(calls):
    """The device time of each call: 20 of it as one graph, the least of 12 replays in turn."""
    graphs = []
    for call in calls:
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            assert call() == 0
            s.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                for _ in range(20):
                    assert call() == 0
        graphs.append(g)
    best = [float("inf")] * len(graphs)
    for _ in range(12):
        for i, g in enumerate(graphs):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            g.replay()
            b.record()
            torch.cuda.synchronize()
            best[i] = min(best[i], 50 * a.elapsed_time(b))
    print(" ".join("%.2f us" % t for t in best))
    return best


def test_operand_of_ragged_rows_costs_what_whole_tiles_do():
    """A row tile's workgroups share its rows in one L2 whatever the number of tiles: 520 rows of 4096 with the norm (33
    tiles) take about the time of 512 (32), not that of every XCD reading every row (1.8 times)."""
    L, K = S.lib(), 4096
    nw, keep, calls = torch.ones(K, device="cuda"), [], []
    for M in (512, 520):
        x, xa = torch.randn(M, K, device="cuda"), U.empty(L.snk_xa_bytes(M, K))
        keep.append((x, xa))
        calls.append(lambda x=x, xa=xa, M=M: L.snk_quant_act(U.ptr(x), M, K, K, U.ptr(nw), 1e-6, U.ptr(xa), U.stream()))
    whole, ragged = least_us(calls)
    assert ragged < 1.45 * whole


def test_added_output_costs_little_more_than_a_stored_one():
    """The many-row kernel's add epilogue loads a tile's output before it stores any of it: 256 rows of 1000 x 1056 added
    take about the time of the same stored, not a load's wait for each of a lane's 16 rows (1.5 times)."""
    L, M, N, K = S.lib(), 256, 1000, 1056
    w, xa, y = U.empty(L.snk_q4_stripes_bytes(N, K)), U.empty(L.snk_xa_bytes(M, K)), U.empty(4 * M * N)
    nb = L.snk_q4_workspace_bytes(M, N, K)
    ws = U.empty(nb)
    store, add = least_us([lambda e=e: L.snk_q4_gemm(U.ptr(w), U.ptr(xa), M, N, K, U.ptr(y), N, e, U.ptr(ws), nb, U.stream())
                           for e in (STORE, ADD)])
    assert add < 1.3 * store


@pytest.mark.parametrize("M,N,K,epi,pad,off", [
    (1, 64, 32, STORE, 0, 0),          # one slice
    (33, 2080, 1024, SWIGLU, 0, 0),    # two slices
    (3, 4, 4096, ADD, 0, 0),           # one thread a row
    (5, 1001, 4096, STORE, 0, 0),      # columns not a multiple of 4: the scalar form
    (7, 1000, 4096, ADD, 3, 0),        # rows of y unaligned: the scalar form
    (7, 1000, 4096, ADD, 4, 0),
    (17, 2560, 9728, STORE, 0, 1),     # y off 16 bytes: the scalar form
    (17, 2560, 9728, ADD, 0, 4),
    (2, 96, 9728, SWIGLU, 0, 0),       # most slices; F = 48
    (2, 96, 9728, SWIGLU, 1, 0),
    (95, 4128, 1056, SWIGLU, 0, 0),    # more than single wavefronts' worth
])
def test_slice_sum_epilogues(M, N, K, epi, pad, off):
    """The slices' sum in its 4-column and scalar forms against 64-bit sums of the same integers and scales. Both sides
    add the same K / 32 products; in 32 bits each of those and the slices' adds rounds once (the scale's product too):
    within (K / 32 + 18) 2^-24 of the sum of their magnitudes; SwiGLU: gate and up so, |silu'| <= 1.1, its own few
    roundings and the exponent's (|g| of them) beside."""
    from oracle import oracle as O

    L, r = S.lib(), np.random.default_rng(M * 11 + N)
    raw = weights(r, N, K, 2)
    w = U.empty(L.snk_q4_stripes_bytes(N, K))
    assert L.snk_q4_repack(U.ptr(U.dev(raw)), N, K, U.ptr(w), U.stream()) == 0
    x = r.standard_normal((M, K)).astype(np.float32)
    ldy = (N // 2 if epi == SWIGLU else N) + pad
    y0 = r.standard_normal(M * ldy + off + 8).astype(np.float32)
    got = matmul(L, 2, w, x, N, epi, ldy, y0, off)
    xa = U.empty(L.snk_xa_bytes(M, K))
    assert L.snk_quant_act(U.ptr(U.dev(x)), M, K, K, None, 1e-6, U.ptr(xa), U.stream()) == 0
    a = U.xa_values(U.host(xa, np.uint8), M, K).astype(np.float64)
    b = O.dequantize_q4_0(raw.reshape(N, -1), K).reshape(N, K).astype(np.float64)
    want, mag = a @ b.T, np.einsum("mbk,nbk->mnb", a.reshape(M, -1, 32), b.reshape(N, -1, 32))
    mag = np.abs(mag).sum(-1) * (K // 32 + 18) * 2.0 ** -24
    if epi == SWIGLU:  # stripes of 16 columns, gate and up in turn
        s, m = want.reshape(M, -1, 2, 16), mag.reshape(M, -1, 2, 16)
        g, u, dg, du = s[:, :, 0], s[:, :, 1], m[:, :, 0], m[:, :, 1]
        sg = g / (1 + np.exp(-g))
        want = (sg * u).reshape(M, -1)
        mag = (1.1 * dg * (np.abs(u) + du) + np.abs(sg) * du + (8 + 2 * np.abs(g)) * 2.0 ** -24 * np.abs(sg * u) + 1e-12).reshape(M, -1)
    y = y0.copy()
    rows = y[off:off + M * ldy].reshape(M, ldy)
    cols = want.shape[1]
    base = rows[:, :cols].astype(np.float64) if epi == ADD else 0.0
    out = got[off:off + M * ldy].reshape(M, ldy)
    assert np.all(np.abs(out[:, :cols] - (want + base)) <= mag + 2.0 ** -23 * np.abs(want + base) + 1e-12)
    keep = np.ones(y.size, bool)
    keep[off:off + M * ldy].reshape(M, ldy)[:, :cols] = False
    assert np.array_equal(got[keep], y[keep])  # nothing past the columns is written


@pytest.mark.parametrize("rows", [191, 200, 255, 257])
def test_step_rows_around_the_many_row_launches(tmp_path, rows):
    """A prompt step whose gate|up (and q|k|v) take the many-row kernel below 256 rows against the same rows in steps of
    40, whose matmuls keep their fused epilogues: every sampled row's logits bit for bit."""
    path = str(tmp_path / "m.gguf")
    S.write_model(path, S.model_cfg(2, 2048, 16, 4, 3584, 1000), 5)
    tok = np.random.default_rng(rows).integers(0, 1000, rows).astype(np.int32)

    sampled = np.array([0, 31, 70, rows // 2, rows - 1])

    def logits(step):
        out = []
        with S.Engine(path, slots=1, ctx=320, max_rows=272) as eng:
            for p in range(0, rows, step):
                n = min(step, rows - p)
                at = sampled[(sampled >= p) & (sampled < p + n)] - p
                eng.step(tok[p:p + n], np.zeros(n, np.int32), np.arange(p, p + n, dtype=np.int32), at, n_write=0)
                if len(at):
                    out.append(eng.logits(np.arange(len(at))))
        return np.concatenate(out)

    assert np.array_equal(logits(rows).view(np.uint32), logits(40).view(np.uint32))


@pytest.mark.parametrize("rows,split", [(192, False), (238, False), (239, True), (255, True)])
def test_rope_epilogue_of_a_narrow_model(tmp_path, rows, split):
    """Q|k|v of a model of width 1024 (4096 x 1024) keeps its RoPE epilogue until the many-row matmul earns the rope
    launch back (1e9 products: 239 rows); the sampled rows' logits are those of steps of 40 either way."""
    path = str(tmp_path / "m.gguf")
    S.write_model(path, S.model_cfg(2, 1024, 16, 8, 3072, 1000), 5)
    tok = np.random.default_rng(rows).integers(0, 1000, rows).astype(np.int32)
    out = []
    for step in (rows, 40):
        with S.Engine(path, slots=1, ctx=320, max_rows=256) as eng:
            for p in range(0, rows, step):
                n = min(step, rows - p)
                eng.prof(step == rows)
                eng.step(tok[p:p + n], np.zeros(n, np.int32), np.arange(p, p + n, dtype=np.int32),
                         np.array([n - 1], np.int32), n_write=0)
            if step == rows:
                assert (eng.prof_read()["rope"]["launches"] > 0) == split
            out.append(eng.logits([0]).copy())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


def test_gate_up_of_a_wide_model_up_to_32_rows(tmp_path):
    """The widest gate|up (51200 columns: enough tiles for the many-row kernel at 24 rows) stays on the streaming kernel
    up to 32 rows, seen without the fused epilogues as one SwiGLU launch more than at 33; the same bits as steps of 11."""
    path = str(tmp_path / "m.gguf")
    S.write_model(path, S.model_cfg(1, 2048, 16, 4, 25600, 1000), 5)
    tok = np.random.default_rng(1).integers(0, 1000, 33).astype(np.int32)
    launches = {}
    with S.Engine(path, slots=40, ctx=64, max_rows=64) as eng:
        eng.graphs(False)
        eng.fuse(False)
        want = None
        for step in (11, 24, 32, 33):
            eng.clear(0, 0, 33)
            out = []
            for p in range(0, 33, step):
                n = min(step, 33 - p)
                eng.prof(True)
                eng.step(tok[p:p + n], np.zeros(n, np.int32), np.arange(p, p + n, dtype=np.int32), np.arange(n), n_write=0)
                launches.setdefault(n, eng.prof_read()["quant"]["launches"])
                eng.prof(False)
                out.append(eng.logits(np.arange(n)).copy())
            got = np.concatenate(out).view(np.uint32)
            want = got if want is None else want
            assert np.array_equal(got, want), step
    assert launches[24] == launches[32] == launches[33] + 1, launches


def test_operand_of_chosen_rows_and_its_normed_rows(tmp_path):
    """The activation quantizer's tile form behind a row list (the LM head's rows of a step) and with the normed rows
    kept (the guess head's input): 800 rows of 400 sequences in one step, 400 of them sampled, against the same in steps
    of 32 rows: logits, and the cells of the model and of its guess head."""
    path = str(tmp_path / "m.gguf")
    S.write_model(path, S.model_cfg(1, 4096, 8, 2, 512, 1000, nextn=1), 5)
    n = 400
    tok = np.random.default_rng(3).integers(0, 1000, (n, 2)).astype(np.int32)
    res = []
    for step in (n, 16):
        with S.Engine(path, slots=n, ctx=64, max_rows=2 * n) as eng:
            assert eng.guess_on(True)
            lg = []
            for s in range(0, n, step):
                seq = np.repeat(np.arange(s, s + step, dtype=np.int32), 2)
                at = 2 * np.arange(step, dtype=np.int32) + (np.arange(s, s + step) % 3 > 0)
                eng.step(tok[s:s + step].reshape(-1), seq, np.tile(np.arange(2, dtype=np.int32), step),
                         at.astype(np.int32), n_write=0)
                lg.append(eng.logits(np.arange(step)).copy())
            res.append((np.concatenate(lg), [eng.kv_save(s, 2).copy() for s in (0, 1, 17, 160, n - 1)]))
    assert np.array_equal(res[0][0].view(np.uint32), res[1][0].view(np.uint32))
    for a, b in zip(res[0][1], res[1][1]):
        assert np.array_equal(a, b)
