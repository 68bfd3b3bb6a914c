"""The one-wave-per-SIMD MLA kernels (csrc/mla_decode_wide.hip): GPU parity with
the oracle at the sizes where they can go wrong -- row counts around the 16, 32,
64 and 128 rows of their variants, pieces around one, two and three tiles (their
ring holds four), shares of many short pieces, second passes in the middle of a
share -- and CPU checks of the generated code.

Tolerance, element by element (that of test_mla.py): weights are rounded to bf16
for the PV product and the output to bf16, each within 2^-9 relative, so |out -
oracle| is at most 2^-8 of the largest value row entry (~4.5 for N(0, 1)):
1.8e-2. That is more than a whole output of many tokens, so each row's error is
also held against the row, 2-norm over 2-norm: independent value rows add the
weights' errors in squares, 2^-9 of the row, and the output's rounding another
2^-9; 1e-2 leaves a factor of 2.5 for value rows that are not.
"""

import os
import re
import shutil
import subprocess

import numpy as np
import pytest
import torch

import capi
from cases import make_mla_case
from test_mla import SCALE, oracle, run, run_balanced
from test_mla import check as check_elements
from test_mla_codegen import HIPCC, ROOT, kernel_body, tile_loops

ROW_REL = 1e-2


def row_errors(out, want):
    """2-norm of each row's error over that of the row (0 for rows of zeros)."""
    off, size = np.linalg.norm(out - want, axis=-1), np.linalg.norm(want, axis=-1)
    return np.where(size > 0, off / np.where(size > 0, size, 1.0), off)


def check(got, want, label):
    check_elements(got, want, label)
    worst = float(row_errors(got[0].float().cpu().numpy(), want[0]).max())
    assert worst <= ROW_REL, f"{label}: a row is {worst:.1e} off"


@pytest.mark.parametrize("S,pieces", [(300, 4), (4096, 59), (9000, 64)])
def test_check_sees_a_lost_tile(S, pieces):
    # What the element-wise tolerance lets pass in long requests: a kernel that
    # leaves a tile out of the PV product, takes the last tile's weights for it,
    # or loses the accumulator of one piece while keeping its sum of weights.
    rng = np.random.default_rng(S)
    q, keys = rng.standard_normal((8, 576)), rng.standard_normal((S, 576))
    p = np.exp(q @ keys.T * SCALE)
    p /= p.sum(axis=1, keepdims=True)
    want = p @ keys[:, :512]
    at = 32 * (S // 64)
    lost, stale, piece = p.copy(), p.copy(), p.copy()
    lost[:, at:at + 32] = 0
    stale[:, at:at + 32] = p[:, at - 32:at]
    piece[:, at:at + S // pieces] = 0
    for wrong in (lost, stale, piece):
        assert row_errors(wrong @ keys[:, :512], want).max() > 2 * ROW_REL
    assert row_errors(want.astype(np.float32), want).max() < 1e-6


EDGES = [1, 31, 32, 33, 0, 63, 64, 65, 95, 96, 97, 128, 129, 161, 300]
# (s_q, h_q): one row; the 16-, 32-, 64- and 128-row variants, full and one
# short or over; a second row group.
ROWS = [(1, 1), (1, 15), (1, 16), (1, 17), (2, 16), (1, 33), (4, 16), (1, 65), (1, 97), (2, 64),
        (1, 129)]


@pytest.mark.gpu
@pytest.mark.parametrize("s_q,h_q", ROWS)
@pytest.mark.parametrize("bs", [32, 64, 96])
def test_rows_and_tile_edges(gpu, s_q, h_q, bs):
    print(f"wide s_q={s_q} h_q={h_q} bs={bs}", flush=True)
    case = make_mla_case(EDGES, s_q, h_q, bs, pool_factor=1.5, seed=h_q + bs, device="cuda",
                         poison=True)
    for causal in {False, s_q > 1}:
        want = oracle(case, causal)
        for nwg in (1, 3, 40, 256):  # one share of every piece ... one tile per share
            check(run_balanced(case, causal, nwg), want, f"bal n{nwg}/c{causal}")
        for ns in (1, 2, 7):
            check(run(case, causal, ns), want, f"ns{ns}/c{causal}")


@pytest.mark.gpu
@pytest.mark.parametrize("s_q,h_q", [(1, 3), (1, 16), (1, 32), (1, 64), (2, 64), (1, 129)])
@pytest.mark.parametrize("bs", [4, 8, 16, 24, 40, 56])  # (4: the per-lane gather)
def test_tiles_over_several_blocks(gpu, s_q, h_q, bs):
    # A tile's four row blocks lie in up to four cache blocks; the last ones past
    # a request's end have no block (their table entries are -1 or the next
    # request's), in first, last and only tiles, and at the table's end.
    lens = EDGES + [7, 8, 9, 15, 16, 17, 23, 24, 25, 39, 40, 41, 302, 311]
    case = make_mla_case(lens, s_q, h_q, bs, pool_factor=1.5, seed=h_q + bs, device="cuda",
                         poison=True)
    for causal in {False, s_q > 1}:
        want = oracle(case, causal)
        for nwg in (1, 3, 40, 256):
            check(run_balanced(case, causal, nwg), want, f"bal n{nwg}/c{causal}")
        for ns in (1, 2, 7):
            check(run(case, causal, ns), want, f"ns{ns}/c{causal}")


@pytest.mark.gpu
@pytest.mark.parametrize("s_q,h_q", [(1, 16), (1, 32), (1, 64), (1, 128)])
def test_second_pass_mid_share(gpu, s_q, h_q):
    # Keys that beat everything else by more than 128 log2 units (fp32 overflows
    # without the second pass), past their piece's first tile, in pieces that
    # follow and precede others of the same share.
    S_list = [40, 700, 33, 300, 95]
    case = make_mla_case(S_list, s_q, h_q, 64, pool_factor=1.5, seed=7, device="cuda", poison=True)
    q, kv, bt, sl = case
    for b, row, tok in ((1, h_q - 1, 405), (1, h_q // 2, 690), (3, 1, 45), (4, 5, 94)):
        kv[int(bt[b, tok // 64]), tok % 64, 0] = (q[b, 0, row].float() * 5).to(torch.bfloat16)
        ids = bt[b, :-(-S_list[b] // 64)].long()
        keys = kv[ids].flatten(0, 1)[:S_list[b], 0].double().cpu()
        sc = (keys @ q[b, 0, row].double().cpu()).numpy() * SCALE / np.log(2.0)
        assert sc[tok] - np.delete(sc, tok).max() > 128.0
    want = oracle(case, False)
    for nwg in (1, 2, 5):
        got = run_balanced(case, False, nwg)
        assert torch.isfinite(got[0].float()).all()
        check(got, want, f"h{h_q}/n{nwg}")
    for ns in (1, 3):
        check(run(case, False, ns), want, f"h{h_q}/ns{ns}")


@pytest.mark.gpu
@pytest.mark.parametrize("S,ns", [(4096, 2), (4160, 2)])
def test_either_side_of_the_split_rule(gpu, S, ns):
    # 2048 tokens per split at 128 rows: either side runs another kernel, and
    # their lse tell which (the 8-wave ones sum rounded weights, 3.6e-6 off in
    # the mean at 4096 tokens; the others are within fp32 rounding). 120
    # requests: the splits alone fill the CUs.
    case = make_mla_case([S] + [70] * 119, 1, 128, 64, seed=S, device="cuda")
    got, want = run(case, False, ns), oracle(case, False)
    check(got, want, f"S{S}/ns{ns}")
    q, kv, bt, _ = case
    keys = kv[bt[0].long()].flatten(0, 1)[:S, 0].double()
    exact = torch.logsumexp(torch.matmul(q[0, 0].double(), keys.t().contiguous()) * SCALE, dim=1)
    off = float((got[1][0, :, 0].double() - exact).norm() / exact.norm())
    assert (off < 5e-7) == (S > 2048 * ns), f"lse {off:.1e} off"


@pytest.mark.gpu
@pytest.mark.parametrize("S_list,s_q,nwg", [([256], 4, 1), ([288], 4, 1), ([128, 128], 8, 2),
                                            ([64], 8, 1), ([1] * 8, 16, 4)])
def test_few_tiles_on_few_workgroups(gpu, S_list, s_q, nwg):
    # Up to 8 tiles and just above at 128 rows per workgroup, several row groups
    # in few shares: one plan for all (the launch leaves the weight of its pieces
    # or, in an even batch, none behind; the 8-wave kernels had other shares).
    case = make_mla_case(S_list, s_q, 128, 64, seed=s_q, device="cuda", poison=True)
    for causal in (False, True):
        check(run_balanced(case, causal, nwg), oracle(case, causal), f"{S_list}/n{nwg}/c{causal}")
    pre, n = launched_plan(case, nwg)
    assert n == 1 and pre[1] == -(-S_list[0] // 32) + 8


@pytest.mark.gpu
@pytest.mark.parametrize("h_q,nwg", [(16, 256), (32, 256), (128, 256), (128, 60), (128, 12),
                                     (128, 2)])
@pytest.mark.parametrize("S_list", [[5, 100, 33], [2100, 700, 64]])
def test_lse_accuracy(gpu, h_q, nwg, S_list):
    # lse sums the weights before their rounding: the largest error here is that
    # of a few fp32 roundings near the value (|lse| < 16: an ulp is 2^-20), where
    # rounded weights are 1e-5 to 1e-3 off. In every row variant, direct and
    # merged.
    case = make_mla_case(S_list, 1, h_q, 64, pool_factor=1.5, seed=h_q, device="cuda", poison=True)
    q, kv, bt, _ = case
    _, lse = run_balanced(case, False, nwg)
    for b, S in enumerate(S_list):
        keys = kv[bt[b, :-(-S // 64)].long()].flatten(0, 1)[:S, 0].double()
        exact = torch.logsumexp(torch.matmul(q[b, 0].double(), keys.t().contiguous()) * SCALE, 1)
        assert float(exact.abs().max()) < 16
        off = float((lse[b, :, 0].double() - exact).abs().max())
        assert off <= 6 * 2.0 ** -20, f"S={S}: {off:.1e} off"


@pytest.mark.gpu
@pytest.mark.parametrize("s_q,h_q", [(1, 30), (1, 60), (1, 128), (2, 65), (3, 128)])
@pytest.mark.parametrize("nwg", [1, 4, 9, 30, 256])
def test_row_groups(gpu, s_q, h_q, nwg):
    # The same batch at every size of row group the rules give it (few
    # workgroups: 128 rows; many: 16), full and ragged groups, causal.
    case = make_mla_case([700, 33, 0, 5, 64, 257], s_q, h_q, 32, pool_factor=1.5, seed=h_q,
                         device="cuda", poison=True)
    want = oracle(case, True)
    check(run_balanced(case, True, nwg), want, f"n{nwg}")
    for ns in (1, 2, 12, 40):
        check(run(case, True, ns), want, f"ns{ns}")


@pytest.mark.gpu
@pytest.mark.parametrize("h_q", [16, 32, 64, 128])
@pytest.mark.parametrize("S,ns,bs", [(16, 1, 64), (70, 2, 64), (200, 3, 64), (70, 2, 12)])
def test_constant_value_column(gpu, h_q, S, ns, bs):
    # A value column that is c in every token is c in the output and in the
    # normalised fp32 states, whatever the weights: both sums of a state add the
    # same weights, c times a bf16 weight is exact in fp32, and a sum of N
    # positive terms is within N 2^-24 of its exact value however it is ordered.
    # (Weights summed before their rounding to bf16: 3e-5 off.) The table is
    # wide enough for fixed splits to take every kernel (12-token blocks: the
    # 8-wave ones).
    q, kv, bt, sl = make_mla_case([S] * 3, 1, h_q, bs, pool_factor=1, seed=S, device="cuda",
                                  poison=True)
    bt = torch.cat([bt, torch.full((3, 8192 // bs), -1, dtype=torch.int32, device="cuda")], 1)
    case = (q, kv, bt.contiguous(), sl)
    cols = {3: 10.0, 200: 1.0, 511: -0.7109375}  # (bf16 values)
    for d, c in cols.items():
        kv[..., d] = torch.where(kv[..., d].isnan(), kv[..., d], c)
    out = torch.empty(3, 1, h_q, 512, dtype=torch.bfloat16, device="cuda")
    lse = torch.empty(3, h_q, 1, dtype=torch.float32, device="cuda")
    wsb = max(capi.mla_workspace_bytes(3, 1, h_q, ns), 16)
    ws = torch.zeros(wsb // 4, dtype=torch.float32, device="cuda")
    assert capi.mla_splitkv_launch(
        q.data_ptr(), kv.data_ptr(), case[2].data_ptr(), sl.data_ptr(), out.data_ptr(),
        lse.data_ptr(), 3, 1, h_q, bs, case[2].shape[1], SCALE, 0, ns, ws.data_ptr(), wsb,
        torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    per_split = -(-(-(-S // ns)) // 32) * 32
    if ns > 1:
        n = 3 * h_q * ns
        acc, l = ws[:n * 512].view(n, 512).double(), ws[n * 513:n * 514].double()
        assert (l > 0).all()
        for d, c in cols.items():
            err = float((acc[:, d] / l / c - 1).abs().max())
            assert err <= (2 * per_split + 4) * 2.0 ** -24, f"state column {d}: {err:.2e} off"
    for got in (run_balanced(case, False, 256)[0], out if ns == 1 else run(case, False, ns)[0]):
        for d, c in cols.items():
            assert (got[..., d].float() == c).all()


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    if not shutil.which(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("mla_wide") / "wide.s"
    csrc = os.path.join(ROOT, "mla-decode-kernels_amd", "csrc")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S",
                    f"-I{os.path.join(ROOT, 'include')}", f"-I{csrc}",
                    os.path.join(csrc, "mla_decode_wide.hip"), "-o", str(out)], check=True,
                   capture_output=True)
    return out.read_text()


def vgprs(text):
    """The VGPR numbers named in an operand list."""
    regs = set()
    for lo, hi in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        regs.update(range(int(lo), int(hi) + 1))
    regs.update(int(x) for x in re.findall(r"\bv(\d+)\b", text))
    return regs


@pytest.mark.parametrize("kernel", ["15mla_wide_kernel", "24mla_wide_balanced_kernel"])
@pytest.mark.parametrize("rw,m,mfmas", [(32, 4, 68), (16, 4, 68), (16, 2, 52), (16, 1, 44)])
def test_generated_tile_loop(asm, kernel, rw, m, mfmas):
    name = f"_ZN3mla12_GLOBAL__N_1{kernel}ILi{rw}ELi{m}EEEvNS_7MlaArgsE"
    body = kernel_body(asm, name)
    # M0 belongs to the copies (inline assembly) alone.
    assert not re.search(r"\bm0\b", re.sub(r";;#ASMSTART.*?;;#ASMEND", "", body, flags=re.S))
    # (The loop over pieces holds the prologue's QK^T as well; the tile loop is
    # the innermost loop that issues MFMAs.)
    shape = "v_mfma_f32_32x32x16_bf16" if rw == 32 else "v_mfma_f32_16x16x32_bf16"
    loops = [t for t in tile_loops(body) if t.count(shape) == mfmas]
    assert len(loops) == 1, "tile loop not found"
    text = loops[0]
    code = [ln for ln in text.split("\n") if ln.strip() and not ln.strip().startswith(";")]
    assert not [ln for ln in code if "scratch_" in ln], "spill access inside the tile loop"
    assert not [ln for ln in code if "v_accvgpr" in ln], "accumulators copied inside the tile loop"
    own = re.sub(r";;#ASMSTART.*?(;;#ASMEND|\Z)", "", text, flags=re.S)
    assert "vmcnt" not in own, "compiler vmcnt wait inside the tile loop"
    # The QK^T results (MFMAs in inline assembly, whose latency the compiler
    # does not know) are not touched before three more MFMAs have issued.
    ops = [ln.split(";")[0].strip() for ln in code]
    qk = [i for i, op in enumerate(ops) if op.startswith(shape + " v[")]
    assert len(qk) == 36
    dst = set()
    for i in qk[-4:]:
        dst |= vgprs(ops[i].split(",")[0])
    later = 0
    for op in ops[qk[-1] + 1:]:
        if op.startswith("v_mfma"):
            later += 1
            if later == 3:
                break
        elif op.startswith(("v_", "ds_", "global_", "buffer_")):
            assert not vgprs(op) & dst, f"QK^T result touched too early: {op}"
    assert later == 3


@pytest.mark.gpu
@pytest.mark.parametrize("bs", [16, 32])
@pytest.mark.parametrize("B", [1, 63, 65, 255, 257, 513, 1100])
def test_plan_of_many_requests(gpu, B, bs):
    # One request per planning thread and several, empty ones in between, at
    # the ends of a wave's lanes too, and shares that start in each of them.
    S_list = [(37 * b) % 71 if b % 5 or b % 64 in (0, 63) else 0 for b in range(B)]
    S_list[-1] = 33
    case = make_mla_case(S_list, 1, 4, bs, pool_factor=1.2, seed=B, device="cuda", poison=True)
    want = oracle(case, False)
    for nwg in (1, 40, 256, 1500):
        check(run_balanced(case, False, nwg), want, f"bal n{nwg}")


@pytest.mark.gpu
@pytest.mark.parametrize("B", [65, 257, 1100])
def test_plan_of_many_requests_gathered(gpu, B):
    # The 8-wave kernel's plan (block sizes off 8).
    test_plan_of_many_requests(gpu, B, 4)


def launched_plan(case, nwg):
    """(the requests' first units and their end [B + 1], shares per row group) of
    a balanced launch, as its split kernel left them behind the states."""
    q, kv, bt, sl = case
    B, s_q, h_q, _ = q.shape
    out = torch.empty(B, s_q, h_q, 512, dtype=torch.bfloat16, device="cuda")
    wsb = capi.mla_balanced_workspace_bytes(B, s_q, h_q, nwg)
    ws = torch.zeros(wsb, dtype=torch.uint8, device="cuda")
    assert capi.mla_balanced_launch(
        q.data_ptr(), kv.data_ptr(), bt.data_ptr(), sl.data_ptr(), out.data_ptr(), None, B, s_q,
        h_q, kv.shape[1], bt.shape[1], SCALE, 0, nwg, ws.data_ptr(), wsb,
        torch.cuda.current_stream().cuda_stream) == 0
    pre = ws[wsb - 8 * (B + 2):].view(torch.int64).cpu()
    return pre[:-1].tolist(), int(pre[-1]) & 0xFFFFFFFF


@pytest.mark.gpu
@pytest.mark.parametrize("B,S,h_q", [(200, 16, 64), (256, 16, 16), (256, 33, 128), (256, 64, 64),
                                     (120, 50, 128), (256, 300, 128)])
def test_a_share_for_every_short_request(gpu, B, S, h_q):
    # Requests that fit the workgroups one each are not put together (a share
    # pays for its pieces one after the other).
    case = make_mla_case([S] * B, 1, h_q, 64, pool_factor=1, seed=S, device="cuda", poison=True)
    want = oracle(case, False)
    check(run_balanced(case, False, 256), want, f"B{B}/S{S}/h{h_q}")
    assert launched_plan(case, 256)[1] >= B


@pytest.mark.gpu
@pytest.mark.parametrize("h_q", [16, 128])
@pytest.mark.parametrize("tiles,nwg,even", [
    ([64, 64], 4, True), ([64] * 3, 3, True), ([65] * 3, 6, True), ([100], 3, True),
    ([64] * 4, 12, True), ([64, 64], 5, False), ([64, 65], 4, False), ([65, 64], 4, False),
    # Not even, for all that the sum, the first and the last one say.
    ([64, 63, 65, 64], 8, False), ([64, 0, 136, 64], 8, False)])
def test_even_batches(gpu, tiles, nwg, even, h_q):
    # Requests of as many tiles each (whatever their last tiles hold) that the
    # shares divide evenly are cut without the weight of a piece, all others
    # with it.
    S_list = [max(0, 32 * t - (7 * i) % 32) for i, t in enumerate(tiles)]
    case = make_mla_case(S_list, 1, h_q, 64, pool_factor=1.5, seed=nwg, device="cuda", poison=True)
    check(run_balanced(case, False, nwg), oracle(case, False), f"{tiles}/n{nwg}/h{h_q}")
    pre, n = launched_plan(case, nwg)
    weight = 0 if even else 8  # kWidePieceCost
    want = [0]
    for t in tiles:
        want.append(want[-1] + (t + weight if t else 0))
    assert pre == want and n == nwg


@pytest.mark.gpu
@pytest.mark.parametrize("s_q,h_q", [(1, 5), (1, 128), (2, 100), (2, 128), (3, 128)])
@pytest.mark.parametrize("S_list", [[511], [512], [4096], [9000, 40], [2000, 1, 0, 700]])
def test_merges(gpu, s_q, h_q, S_list):
    # Rows of few and of many pieces (from 16 on, up to 256 rows: 16 waves a
    # row; else a wave a row), rows off the four of a workgroup, and requests
    # that are not cut at all.
    case = make_mla_case(S_list, s_q, h_q, 64, pool_factor=1.5, seed=h_q, device="cuda",
                         poison=True)
    want = oracle(case, False)
    for nwg in (40, 256):
        first = run_balanced(case, False, nwg)
        check(first, want, f"bal n{nwg}")
        again = run_balanced(case, False, nwg)
        assert torch.equal(first[0], again[0]) and torch.equal(first[1], again[1])
    for ns in (3, 15, 16, 17, 64):
        check(run(case, False, ns), want, f"ns{ns}")
