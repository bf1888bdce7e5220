"""The round-4 prefill paths against the paths they replace, on ONE library build (the switches are read once per process, so every leg is its own
process running tools/ab_prefill_bits.py: a 700-token prefill + 8 greedy tokens of a DeltaNet + attention model at model_dim 1024):

  * four-channel conv apply (k_deltanet.hip::conv_apply4_kernel)                  -- BIT-IDENTICAL logits to the one-channel kernel
  * split-K reduction + Normalization in one launch (normalization_from_partials)  -- BIT-IDENTICAL logits, fewer launches
  * DeltaNet scan as two concurrent segments (k_deltanet_chunk.hip: ScanSplit)     -- another summation order: logits within the parity tolerance
  * DeltaNetPrefillPrep inside the chunk preparation (round 6: dn_chunk_prep_kernel<true>) -- BIT-IDENTICAL logits to the two launches, fewer launches
  * the head norms inside the AttentionPrepare launch, SigmoidGate inside the key-split merge (round 6)  -- BIT-IDENTICAL logits, fewer launches
  * the conv out of place without its halo launch (round 6: conv_apply4_oop_kernel)          -- BIT-IDENTICAL logits (and the same carried conv state: the decode steps
                                                                                              behind the prefill produce the same tokens)
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from helpers import f32

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _leg(tmp_path, name, args=("--prompt", "700"), **env):
    dump = str(tmp_path / f"{name}.npy")
    out = subprocess.run([sys.executable, os.path.join(ROOT, "tools", "ab_prefill_bits.py"), "--model", "tiny", *args, "--dump", dump],
                         env=dict(os.environ, **env), capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    rec = json.loads(out.stdout.strip().splitlines()[-1])
    rec["logits"] = np.load(dump)
    return rec


def test_prefill_switches_bit_identity_and_tolerance(tmp_path):
    base = _leg(tmp_path, "default")
    conv1 = _leg(tmp_path, "conv1", UZU_HIP_TUNE="conv_apply4=0")
    two = _leg(tmp_path, "two_launches", UZU_HIP_TUNE="norm_partials=0")
    chain = _leg(tmp_path, "one_chain", UZU_HIP_TUNE="dn_split=0")
    prep = _leg(tmp_path, "prep_launch", UZU_HIP_TUNE="prep_fused=0")  # DeltaNetPrefillPrep as its own launch in front of the chunk preparation
    assert prep["logits_sha256"] == base["logits_sha256"] and prep["tokens"] == base["tokens"]
    assert prep["prefill_launches"] > base["prefill_launches"], (prep["prefill_launches"], base["prefill_launches"])
    attn = _leg(tmp_path, "attn_separate", UZU_HIP_TUNE="attn_fused=0")  # QKVNorm launches in front of AttentionPrepare, SigmoidGate behind the attention merge
    assert attn["logits_sha256"] == base["logits_sha256"] and attn["tokens"] == base["tokens"]
    assert attn["prefill_launches"] > base["prefill_launches"], (attn["prefill_launches"], base["prefill_launches"])
    inplace = _leg(tmp_path, "conv_in_place", UZU_HIP_TUNE="conv_oop=0")  # the conv in place behind its halo launch instead of out of place
    assert inplace["logits_sha256"] == base["logits_sha256"] and inplace["tokens"] == base["tokens"]
    assert conv1["logits_sha256"] == base["logits_sha256"] and conv1["tokens"] == base["tokens"]
    assert two["logits_sha256"] == base["logits_sha256"] and two["tokens"] == base["tokens"]
    assert two["prefill_launches"] > base["prefill_launches"], (two["prefill_launches"], base["prefill_launches"])  # the fused path really ran
    # the split scan: f32 sums in another order in front of a bf16 rounding, then three more layers: the logits stay within 0.05 sigma of the one-chain scan
    a, b = f32(base["logits"]).astype(np.float64), f32(chain["logits"]).astype(np.float64)
    assert np.abs(a - b).max() <= 0.05 * b.std(), (np.abs(a - b).max(), b.std())
    assert chain["first_token"] == base["first_token"]


def test_split_products_of_dozens_of_rows_end_in_the_next_normalization(tmp_path):
    """The same for a prompt whose down projections run in the register-fed kernel with K split (csrc/k_gemm_rows.hip; K of 2048 in groups of 128): the launch that adds the shares and
    normalises against the two launches it replaces."""
    args = ("--prompt", "70", "--hidden", "2048", "--group", "128")
    base = _leg(tmp_path, "rows", args)
    two = _leg(tmp_path, "rows_two_launches", args, UZU_HIP_TUNE="norm_partials=0")
    assert two["logits_sha256"] == base["logits_sha256"] and two["tokens"] == base["tokens"]
    assert two["prefill_launches"] > base["prefill_launches"], (two["prefill_launches"], base["prefill_launches"])


@pytest.mark.parametrize("prompt,hidden", [(4, 2048), (13, 3584), (16, 2176)])
def test_few_rows_share_k_in_front_of_a_normalization(tmp_path, prompt, hidden):
    """A few rows' down projections (csrc/k_gemv_rows.hip) in shares of K -- equal ones, and 17 or 28 steps in four -- which the next Normalization adds, against whole sums.  Another order of
    f32 sums flips a bf16 rounding in 2e4 (2^-23 of a value against its 2^-8 steps), and one flip moves some logit of this model by up to 0.1 sigma, so the legs are not held against each other but
    each against the reference-order pass: as close as the whole sums (RMS; a quarter for the flips, 7 % seen)."""
    args = ("--prompt", str(prompt), "--hidden", str(hidden), "--group", "128")
    shares = _leg(tmp_path, "shares", args)
    whole = _leg(tmp_path, "whole", args, UZU_HIP_TUNE="norm_partials=0")
    assert whole["prefill_launches"] > shares["prefill_launches"], (whole["prefill_launches"], shares["prefill_launches"])
    exact, a, b = (f32(r["logits"]).astype(np.float64) for r in (_leg(tmp_path, "exact", args, UZU_HIP_EXACT="1"), shares, whole))
    rms = lambda d: np.sqrt((d ** 2).mean())
    assert rms(a - exact) <= 1.25 * rms(b - exact), (rms(a - exact), rms(b - exact), exact.std())


@pytest.mark.parametrize("dim", [1024, 2048, 4096])
def test_rows_in_pair_order_leave_the_logits_as_they_are(tmp_path, dim):
    """Normalizations and the gated epilogue write their rows in the order that the DMA form of the int4 products reads (csrc/k_gemm_dma.hip), a thread's 4, 8 or 16 elements at a
    time; the wave-specialised form takes plain rows.  The MLP is wider than 4096, so both legs sum a row's groups in the same order: the same bits."""
    args = ("--prompt", "300", "--dim", str(dim), "--hidden", "4352", "--group", "128")
    plain = _leg(tmp_path, "plain", args, UZU_HIP_TUNE="gemm_form=2")
    for form in ("0", "1"):
        pairs = _leg(tmp_path, f"pairs{form}", args, UZU_HIP_TUNE=f"gemm_form={form}")
        assert pairs["logits_sha256"] == plain["logits_sha256"] and pairs["tokens"] == plain["tokens"], form


def test_producers_write_the_rows_in_pair_order(tmp_path):
    """The same bits come from the copy that a product's pre-pass makes of plain rows: that the producers wrote them shows in the first pass's memory, the workspace without the copy of the
    down projection's 1021 x 16384 rows (33 MB; 38 and 70 MiB seen)."""
    args = ("--prompt", "1021", "--hidden", "16384", "--group", "128")
    pairs = _leg(tmp_path, "pairs", args, UZU_HIP_TUNE="gemm_form=0")
    assert pairs["first_pass_bytes"] < 55 << 20, pairs["first_pass_bytes"]


@pytest.mark.parametrize("prompt,dim,hidden", [(520, 4096, 4352), (449, 4096, 4096)])
def test_gated_rows_in_pair_order_reach_the_form_that_reads_them(tmp_path, prompt, dim, hidden):
    """Down projections just above the staged kernel's count of tiles (csrc/k_gemm_rows.hip), with their choice of kernel unpinned: gated rows exist in pair order only, and a product that
    did not take them would fail the pass.  Other products of the pass sum in other orders than those of plain rows on one form, and a flipped rounding of the residual rows moves logits by
    up to 0.14 sigma here, so each is held against the reference-order pass: as close as plain rows (RMS; a quarter for the flips, as above)."""
    args = ("--prompt", str(prompt), "--dim", str(dim), "--hidden", str(hidden), "--group", "128")
    legs = _leg(tmp_path, "exact", args, UZU_HIP_EXACT="1"), _leg(tmp_path, "auto", args), _leg(tmp_path, "plain", args, UZU_HIP_TUNE="gemm_form=2")
    exact, a, b = (f32(r["logits"]).astype(np.float64) for r in legs)
    rms = lambda d: np.sqrt((d ** 2).mean())
    assert rms(a - exact) <= 1.25 * rms(b - exact), (rms(a - exact), rms(b - exact), exact.std())
