"""The attention output block (pcl_attention_output): projection, post-norm
and residual, src/engine/attention.rs:866-884.

CPU tests pin the oracle's p9_ref_matvec and p9_ref_add restatements with the
reference's known answers (src/kernels/reference/tests.rs:14-19, 67-73) and
with the f64-accumulation property the reference tests for its projections
(tests.rs:21-47: 2^24 + 1 - 2^24 keeps the 1). GPU tests compare the
projection kernels (a wave per row; f64 MFMAs for few tokens; f64 MFMA tiles)
and the fused post-norm with the oracle.
"""
import numpy as np
import pytest

from helpers import normals


# ---- oracle pinning (CPU) --------------------------------------------------

def test_matrix_orientation_is_output_rows_by_input_columns(oracle):
    # src/kernels/reference/tests.rs:14-19
    y = oracle.matvec([1.0, 2.0, 3.0, -1.0, 0.0, 2.0], [1.0, 2.0, 4.0], 2, 3)
    assert y.tolist() == [17.0, 7.0]


def test_projection_accumulates_in_f64(oracle):
    # the property of tests.rs:21-47: an f32 sum would lose the 1
    y = oracle.matvec([16777216.0, 1.0, -16777216.0], [1.0, 1.0, 1.0], 1, 3)
    assert y.tolist() == [1.0]


def test_add_and_block_composition(oracle):
    # tests.rs:67-73, then the block: residual + rms_norm(W x) (attention.rs:
    # 866-884) against an independent f64 restatement
    assert oracle.add([2.0], [3.0]).tolist() == [5.0]
    rows, cols = 48, 64
    w = normals(1, rows * cols) * np.float32(0.1)
    x = normals(2, cols)
    scale = normals(3, rows)
    res = normals(4, rows)
    proj, out = oracle.attention_output(x, w, scale, 1e-6, res, rows, cols)
    want_p = (w.reshape(rows, cols).astype(np.float64) @ x.astype(np.float64)).astype(np.float32)
    assert np.array_equal(proj, want_p)
    p64 = proj.astype(np.float64)
    inv = 1.0 / np.sqrt(np.mean(p64 * p64) + 1e-6)
    want = (res + (p64 * inv).astype(np.float32) * scale).astype(np.float32)
    assert np.max(np.abs(out - want)) <= 1e-6


# ---- the device output block (GPU) -----------------------------------------

@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a GPU"
    return t


@pytest.fixture(scope="module")
def ctx(pcl, torch):
    c = pcl.Context(0, torch.cuda.current_stream().cuda_stream)
    yield c
    c.close()


def dev(torch, x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to("cuda:0")


def run_block(torch, ctx, x, w, scale, res, eps=1e-6, in_place=False):
    n, cols = x.shape
    rows = w.shape[0]
    tx, tw, ts, tr = dev(torch, x), dev(torch, w), dev(torch, scale), dev(torch, res)
    proj = torch.full((n, rows), float("nan"), device="cuda:0")
    out = tr if in_place else torch.full((n, rows), float("nan"), device="cuda:0")
    ctx.attention_output(tx.data_ptr(), n, cols, tw.data_ptr(), rows, ts.data_ptr(), eps,
                         tr.data_ptr(), proj.data_ptr(), out.data_ptr())
    err = ctx.sync()
    return proj.cpu().numpy(), out.cpu().numpy(), err


# n = 1 and 5: a wave per output row; 7, 16, 17, 32: the few-token kernel; 33,
# 200, 300: a wave per 16 x 16 block. One token
# with input rows of at most 16384 columns (a multiple of 4) is projected
# with the input row staged in LDS: rows of 1000 (fewer than 4096 columns),
# 5000 (4096 and a partial step), 4000 (one 4096-column step taken by some
# lanes only) and 4096 columns; 16388 and 1001
# columns take the plain one-token kernel.
BLOCK_CASES = [(1, 4096, 2816), (5, 4096, 2816), (16, 8192, 2816), (32, 4096, 1536),
               (33, 4096, 2816), (200, 4096, 300), (300, 1000, 130), (7, 1001, 77),
               (1, 1000, 77), (1, 5000, 300), (1, 4000, 300), (17, 4096, 300),
               (1, 16388, 64), (1, 1001, 77)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", BLOCK_CASES, ids=lambda c: "x".join(map(str, c)))
def test_output_block_matches_the_oracle(torch, ctx, oracle, case):
    n, cols, rows = case
    g = np.random.default_rng(sum(case))
    x = g.standard_normal((n, cols)).astype(np.float32)
    w = (g.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32)
    scale = (1 + 0.1 * g.standard_normal(rows)).astype(np.float32)
    res = g.standard_normal((n, rows)).astype(np.float32)
    proj, out, err = run_block(torch, ctx, x, w, scale, res)
    assert err == 0
    same = 0
    for t in range(n):
        want_p, want = oracle.attention_output(x[t], w, scale, 1e-6, res[t], rows, cols)
        # f64 sums in another order: equal unless an f32 rounding boundary
        # falls between the two f64 sums (relative 1e-15 apart)
        assert np.max(np.abs(proj[t] - want_p) / (1e-30 + np.abs(want_p))) <= 2 ** -23
        assert np.max(np.abs(out[t] - want)) <= 1e-5
        same += int(np.sum(proj[t].view(np.uint32) == want_p.view(np.uint32)))
    assert same >= 0.999 * n * rows


# (tokens, columns, output rows) and the form they take on 256 CUs: a wave per
# output row (1), the few-token kernel with 16 or 32 tokens a workgroup, a
# wave per 16 x 16 block (16016: columns below, at and past its groups of 16
# and its 16 groups in flight), or output tiles of tokens x rows (tokens *
# 1000 + rows). Per tile shape: a remainder of tokens and rows, columns below
# one K step, and more than two K steps with a remainder. The few-token
# kernel: one to 32 tokens around its blocks of 16, output rows of 16 and one
# past, columns within one wave's 16, at and past 256-column steps, and
# remainders of a quad; enough rows for two blocks a workgroup.
FORMS = {
    (3, 4, 1): 1, (4, 28, 16): 1, (5, 4096, 2816): 1, (3, 1001, 77): 1, (5, 1003, 33): 1,
    (6, 4, 1): 16, (13, 1001, 77): 16, (16, 260, 17): 16, (17, 256, 33): 16, (31, 126, 32): 16,
    (17, 127, 33): 16, (32, 516, 16): 16, (31, 770, 4100): 32, (32, 1024, 2816): 32,
    (33, 3, 17): 16016, (33, 512, 40): 16016, (40, 130, 65): 16016, (48, 16, 129): 16016,
    (64, 1028, 31): 16016, (65, 772, 33): 16016, (80, 277, 2816): 16016, (128, 96, 18): 16016,
    (81, 381, 2811): 32032, (129, 68, 2816): 32032, (200, 381, 2816): 32032, (65, 96, 4220): 32032,
    (530, 34, 4220): 64032, (480, 200, 2816): 64032, (497, 261, 2801): 64032,
    (700, 63, 2816): 64064, (700, 330, 2816): 64064, (300, 199, 2803): 64064,
    (520, 65, 2816): 128064, (2100, 101, 2816): 128064, (1400, 31, 2816): 128128,
    (1400, 133, 2816): 128128, (1301, 98, 2790): 128128,
}


def test_projection_forms(pcl):
    form = pcl.load().pcl_debug_projection_form
    for case, want in FORMS.items():
        assert form(*case, 256) == want, case
    # the column count decides between shapes: whole K steps of 32 for narrow
    # rows (2000 x 96: 39 us in 128 x 64, 49 us in 64 x 32), less padding of
    # tokens for wide ones
    assert form(2000, 96, 2816, 256) == 128064 and form(2000, 4096, 2816, 256) == 64032
    assert form(520, 64, 2816, 256) in (64064, 64032, 128064)
    assert form(1, 4096, 2816, 256) == 1 and form(33, 4096, 2816, 0) // 1000 >= 32
    # one chain per SIMD, or tiles
    assert form(80, 4096, 2816, 256) == 16016 and form(81, 4096, 2816, 256) == 32032
    assert form(48, 4096, 2816, 256) == 16016 and form(64, 4096, 2816, 256) == 32032
    # sizes at the entry's limits stay within a grid's 65535 blocks of rows
    assert form(1 << 22, 1 << 20, 1 << 20, 256) == 128128
    for n, out in ((1 << 22, 16), (1 << 22, 1 << 20), (1 << 20, 128)):
        assert n / (form(n, 64, out, 256) // 1000) <= 65535


@pytest.mark.gpu
@pytest.mark.parametrize("case", FORMS, ids=lambda c: "x".join(map(str, c)))
def test_projection_matches_f64_sums(torch, ctx, case):
    n, cols, rows = case
    g = np.random.default_rng(sum(case))
    x = g.standard_normal((n, cols)).astype(np.float32)
    w = (g.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32)
    scale = (1 + 0.1 * g.standard_normal(rows)).astype(np.float32)
    res = g.standard_normal((n, rows)).astype(np.float32)
    proj, out, err = run_block(torch, ctx, x, w, scale, res)
    assert err == 0
    p64 = x.astype(np.float64) @ w.astype(np.float64).T
    # one rounding to f32, and f64 sums of `cols` terms in another order
    slack = 2.0 ** -24 * np.abs(p64) + cols * 2.0 ** -52 * (np.abs(x).astype(np.float64)
                                                            @ np.abs(w).astype(np.float64).T)
    assert np.all(np.abs(proj - p64) <= slack)
    q64 = proj.astype(np.float64)
    want = res + (q64 / np.sqrt(np.mean(q64 * q64, axis=1, keepdims=True) + 1e-6)) * scale
    assert np.max(np.abs(out - want)) <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [1000, 3848, 4000, 4092, 4096, 5000, 16384])
def test_one_token_projection_equals_the_multi_token_one_bitwise(torch, ctx, cols):
    # the one-token kernel (input row staged in LDS) sums each row's f64
    # products in the order of the multi-token row kernel
    rows = 300
    g = np.random.default_rng(cols)
    x = g.standard_normal((2, cols)).astype(np.float32)
    w = (g.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32)
    scale = (1 + 0.1 * g.standard_normal(rows)).astype(np.float32)
    res = g.standard_normal((2, rows)).astype(np.float32)
    proj2, out2, err2 = run_block(torch, ctx, x, w, scale, res)
    proj1, out1, err1 = run_block(torch, ctx, x[1:], w, scale, res[1:])
    assert err1 == 0 and err2 == 0
    assert np.array_equal(proj1[0].view(np.uint32), proj2[1].view(np.uint32))
    assert np.array_equal(out1[0].view(np.uint32), out2[1].view(np.uint32))


# A token's projection is the same f64 sum, in one order, in every launch of up
# to 32 tokens, and in one order in every larger one. Columns: below one quad,
# whole 256-column steps and one quad past, remainders of one to three columns,
# more than one 4096-column step, a lone 256-column step; output rows of 16 and
# one past, enough of them for two 16-token blocks a workgroup. Past 32 tokens:
# remainders of tokens, rows and columns in tiles of several shapes, each over
# more than two K steps. The terms of a row cancel in pairs but for a few small
# ones, so that f64 sums in another order differ in their f32 bits.
@pytest.mark.gpu
@pytest.mark.parametrize("case", [(3, 4096, 300), (2, 1001, 33), (4, 1000, 300), (5, 8193, 16),
                                  (6, 1028, 33), (8, 4098, 17), (16, 260, 64), (16, 1, 1),
                                  (17, 4096, 130), (31, 1003, 48), (32, 512, 4200),
                                  (17, 259, 2816), (32, 3, 4200), (34, 4097, 33), (64, 1028, 300),
                                  (128, 196, 65), (96, 260, 2816), (200, 1000, 2816),
                                  (480, 200, 2816), (520, 515, 2816), (700, 261, 2816),
                                  (1400, 133, 2816), (2100, 130, 2816)],
                         ids=lambda c: "x".join(map(str, c)))
def test_a_tokens_projection_does_not_depend_on_the_token_count(torch, ctx, case):
    n, cols, rows = case
    g = np.random.default_rng(sum(case))
    h = cols // 2
    x = (g.standard_normal((n, cols)) * 2.0 ** g.integers(-12, 13, (n, cols))).astype(np.float32)
    w = (g.standard_normal((rows, cols)) * 2.0 ** g.integers(-12, 13, cols)).astype(np.float32)
    order = g.permutation(cols)
    x[:, order[h:2 * h]] = x[:, order[:h]]
    w[:, order[h:2 * h]] = -w[:, order[:h]]
    w[:, order[:h // 8]] += np.float32(1e-6)
    scale = (1 + 0.1 * g.standard_normal(rows)).astype(np.float32)
    res = g.standard_normal((n, rows)).astype(np.float32)
    proj, out, err = run_block(torch, ctx, x, w, scale, res)
    assert err == 0
    few = 1 if n <= 32 else 33
    for t in sorted({0, (n - few) // 2, n - few}):
        rows_t = slice(t, t + few)
        proj1, out1, err1 = run_block(torch, ctx, x[rows_t], w, scale, res[rows_t])
        assert err1 == 0
        assert np.array_equal(proj[rows_t].view(np.uint32), proj1.view(np.uint32))
        assert np.array_equal(out[rows_t].view(np.uint32), out1.view(np.uint32))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 40])
def test_output_block_keeps_f64_cancellation_and_runs_in_place(torch, ctx, oracle, n):
    cols, rows = 96, 40
    x = np.ones((n, cols), np.float32)
    w = np.zeros((rows, cols), np.float32)
    w[:, 0], w[:, 1], w[:, 2] = 16777216.0, 1.0, -16777216.0
    w[:, 3:] = np.float32(1e-3)
    scale = np.ones(rows, np.float32)
    res = normals(5, n * rows).reshape(n, rows)
    proj, out, err = run_block(torch, ctx, x, w, scale, res.copy(), in_place=True)
    assert err == 0
    want_p, want = oracle.attention_output(x[0], w, scale, 1e-6, res[0], rows, cols)
    # the 1 survives (1 + 93e-3, where an f32 sum gives 93e-3); the small
    # terms the MFMA path adds while its partial sum is at 2^24 may move the
    # f32 result by an ulp
    assert np.all(np.abs(proj - 1.093) < 1e-3)
    assert np.max(np.abs(proj - want_p[None, :])) <= 2 ** -23 * 1.1
    assert np.max(np.abs(out - want[None, :] + res[0][None, :] - res)) <= 1e-6


@pytest.mark.gpu
def test_output_block_rejects_bad_arguments_and_flags_non_finite(pcl, torch, ctx):
    x = torch.ones((2, 64), device="cuda:0")
    w = torch.ones((8, 64), device="cuda:0")
    s = torch.ones(8, device="cuda:0")
    r = torch.ones((2, 8), device="cuda:0")
    out = torch.empty((2, 8), device="cuda:0")
    with pytest.raises(pcl.AttentionError) as e:
        ctx.attention_output(x.data_ptr(), 0, 64, w.data_ptr(), 8, s.data_ptr(), 1e-6,
                             r.data_ptr(), out.data_ptr(), out.data_ptr())
    assert e.value.kind == "InvalidShape"
    with pytest.raises(pcl.AttentionError) as e:
        ctx.attention_output(x.data_ptr(), 2, 64, w.data_ptr(), 8, s.data_ptr(), 0.0,
                             r.data_ptr(), out.data_ptr(), out.data_ptr())
    assert e.value.kind == "InvalidParameter"
    x[1, 3] = float("inf")
    proj = torch.empty((2, 8), device="cuda:0")
    ctx.attention_output(x.data_ptr(), 2, 64, w.data_ptr(), 8, s.data_ptr(), 1e-6,
                         r.data_ptr(), proj.data_ptr(), out.data_ptr())
    assert ctx.sync() == 8
