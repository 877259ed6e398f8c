"""GEMM2 from activations held as e4m3 pairs: the form that the sort chooses
at prefill sizes where the experts' slots fill 256-row tiles."""
from __future__ import annotations

import pytest
import torch

from flashinfer_amd import workloads as W
from flashinfer_amd.shapes import DEFINITIONS
from _helpers import log, oracle_subset, run_gpu

pytestmark = pytest.mark.gpu

SMALL = DEFINITIONS[3]  # 16 of 128 experts, top-6, H = 4096, I = 1536


def _all_on_first(T, seed):
    """Every token on the shard's first top_k experts: T rows each."""
    wl = W.make_for(SMALL, f"pairs_{T}", T, seed, local_expert_offset=16)
    wl.tensors["routing_logits"][:, 16:16 + SMALL.TOPK] += 12.0
    return wl


def _choice(T):
    from flashinfer_amd import _lib, kernel
    L = _lib.workspace_layout(T, SMALL)
    return int(kernel.last_workspace()[L.expert_off:L.expert_off + 260 * 4].view(torch.int32)[257])


# Rows of the experts' last tile around what the tile does differently: 32 and 64
# rows a wave group in tiles of at most 128, 64 and 128 rows of the second group
# above, and full tiles only.
@pytest.mark.parametrize("rem", [0, 1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 191, 192,
                                 193, 255])
def test_pair_tile_row_edges(rem, monkeypatch):
    """The first, some inner and the last 24 rows of every expert against the
    oracle, and a normwise error at the bf16 rows' and output's rounding: pairs
    keep 2^-9 of a value (bf16 2^-8), so it is below the 2.9e-3 of bf16
    activations with bf16 rows."""
    from oracle import ref_moe as R
    T = 2816 + rem
    log(f"test_pair_tile_row_edges[{T}]")
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    wl = _all_on_first(T, 5000 + rem)
    out = run_gpu(wl, fill=float("nan"))
    assert _choice(T) == 1
    assert torch.isfinite(out.float()).all()
    tokens = torch.cat([torch.arange(4), torch.arange(250, 262), torch.arange(T - 24, T)])
    rep = R.tolerance_report(out[tokens.cuda()].float().cpu(), oracle_subset(wl, tokens).acc)
    assert rep["n_bad"] == 0, rep
    assert rep["normwise_rel"] <= 2.9e-3, rep


def test_bf16_kept_where_tiles_stay_empty(monkeypatch):
    """Evenly routed tokens leave most rows of 256-row tiles empty: the call is
    bitwise the one with bf16 activations, and within the bar."""
    from oracle import ref_moe as R
    log("test_bf16_kept_where_tiles_stay_empty")
    T = 2740
    wl = W.make_for(SMALL, "even", T, 77)
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    out = run_gpu(wl, fill=float("nan")).clone()
    choice = _choice(T)
    monkeypatch.setenv("MI_MOE_VARIANT", "18,21")  # bf16 activations always
    bf16 = run_gpu(wl, fill=float("nan"))
    tokens = torch.arange(0, T, 97)
    rep = R.tolerance_report(out[tokens.cuda()].float().cpu(), oracle_subset(wl, tokens).acc)
    assert rep["n_bad"] == 0, rep
    assert choice == 0
    assert torch.equal(out.view(torch.int16), bf16.view(torch.int16))


@pytest.mark.parametrize("scale", [float("nan"), float("inf"), 3e33, 1e-36, 0.0])
def test_pairs_nonfinite_and_extreme_rows(scale, monkeypatch):
    """A token whose activations are not finite, overflow, vanish or are zero:
    its output is finite, infinite or NaN where the bf16 form's is, and no other
    token's output changes."""
    log(f"test_pairs_nonfinite_and_extreme_rows[{scale}]")
    T, t = 2816, 300
    wl = _all_on_first(T, 6000)
    monkeypatch.delenv("MI_MOE_VARIANT", raising=False)
    plain = run_gpu(wl).clone()
    wl.tensors["hidden_states_scale"][:, t] = scale
    out = run_gpu(wl).clone()
    assert _choice(T) == 1
    monkeypatch.setenv("MI_MOE_VARIANT", "18,21")
    bf16 = run_gpu(wl)
    others = torch.arange(T, device="cuda") != t
    assert torch.equal(out[others].view(torch.int16), plain[others].view(torch.int16))
    a, b = out[t].float(), bf16[t].float()
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.isinf(a), torch.isinf(b))
    fin = torch.isfinite(b)
    # both forms round act, rows and output: a few bf16 ulps of the row's largest
    assert (a[fin] - b[fin]).abs().max().item() <= 2e-2 * b[fin].abs().max().item() if fin.any() else True
