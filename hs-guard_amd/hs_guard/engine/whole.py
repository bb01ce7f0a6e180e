"""Complete-message scoring on the MI355X kernels: one forward over a whole token sequence.

Replaces the reference's whole forward behind ``score_messages`` (src/hs_guard/runtime.py:136-145): the
Qwen3.5 backbone with FLA's ``chunk_gated_delta_rule`` in the GDN layers (runtime.py:76-89) and the tiled
512-token window attention (src/hs_guard/window_attention.py:34-53, 56-72) in the attention layers, then both
roles' risk heads (runtime.py:71-74).

* GDN layers: fused projection GEMM -> causal conv + SiLU from a zero history -> ``hsg_gdn_chunk_prefill`` from a
  zero state (the WY/UT chunk form on MFMA) -> ``hsg_gated_rmsnorm`` -> out_proj.
* Attention layers: fused q|k|v GEMM -> q/k RMSNorm + RoPE at positions 0 .. T-1 -> ``hsg_window_attention`` (the
  window mask 0 <= p <= q, p > q - W over the sequence's own keys, gated by sigmoid(gate)) -> o_proj.
* Risk heads in float32, as the reference's readout on ``hidden.float()`` outside autocast (runtime.py:70-73,
  141): an fp32 GEMM with the heads' fp32 weights, then ``hsg_risk_head_f32`` (LayerNorm, SiLU, logits and
  softmax, nothing rounded to bf16).

No per-slot state of the streaming engine is read or written.

GEMMs run at the whole sequence's M, so results differ from the streaming path's in the last bits of some
products; the two agree within the tolerances the tests state (the reference's own stream-vs-whole check
allows 0.05, examples/demo/server.py:483).
"""
from __future__ import annotations

import torch

from .._lib import calls, check, lib
from .slot_engine import ROLES, PreparedWeights, gdn_proj_width

SEG = 64                  # query tokens of an attention segment
MAX_ATT_SEGMENTS = 1 << 17    # segments per attention launch: bounds its grid for sequences of millions of tokens


def fp32_heads(model, roles=ROLES):
    """Both roles' risk heads for the complete-message readout, float32 and unrounded (runtime.py:70-73): the first
    Linear fused over the roles (w1 [roles*E, hidden], b1), the LayerNorm (ln_w, ln_b [roles, E]) and the risk
    Linear (w2 [roles, 3, E], b2 [roles, 3])."""
    m, f32 = model, torch.float32
    return {"w1": torch.cat([m[f"heads.{r}.projection.0.weight"] for r in roles]).to(f32).contiguous(),
            "b1": torch.cat([m[f"heads.{r}.projection.0.bias"] for r in roles]).to(f32).contiguous(),
            "ln_w": torch.stack([m[f"heads.{r}.projection.1.weight"] for r in roles]).to(f32).contiguous(),
            "ln_b": torch.stack([m[f"heads.{r}.projection.1.bias"] for r in roles]).to(f32).contiguous(),
            "w2": torch.stack([m[f"heads.{r}.risk.weight"] for r in roles]).to(f32).contiguous(),
            "b2": torch.stack([m[f"heads.{r}.risk.bias"] for r in roles]).to(f32).contiguous()}


class WholeSequenceScorer(PreparedWeights):
    """Scores whole token sequences with the kernels of libhsg.so. ``shared``: a SlotStreamEngine (or another
    scorer) whose prepared weights are reused instead of building a second copy."""

    def __init__(self, model, roles=ROLES, shared=None):
        lib()  # fail loudly if the HIP library is missing
        self.model, self.cfg = model, model.config
        self.roles = tuple(roles)
        self.device = model.device
        types = list(self.cfg.layer_types)
        self.kind = [(t, sum(1 for u in types[:i] if u == t)) for i, t in enumerate(types)]
        self.window = self.cfg.window_tokens
        if shared is not None and tuple(shared.roles) == self.roles:
            for name in ("layers", "final_w1", "emb", "inv_freq", "head_w1", "head_b1", "head_ln_w", "head_ln_b",
                         "head_w2", "head_b2"):
                setattr(self, name, getattr(shared, name))
        else:
            self._prepare_weights()
        self.head32 = fp32_heads(model, self.roles)

    @torch.inference_mode()
    def forward(self, ids):
        """Class probabilities of every position of the token sequence ``ids``: float32 [roles, T, 3] on the
        device (the softmax of each role's risk head)."""
        L = calls()
        cfg, dev = self.cfg, self.device
        T = len(ids)
        if T == 0:
            raise ValueError("The sequence is empty")
        st = torch.cuda.current_stream(dev).cuda_stream
        bf16 = torch.bfloat16
        H, eps, W = cfg.hidden_size, cfg.rms_norm_eps, self.window
        hq, hkv, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
        G = hq // hkv
        nh, hv, kd, vd = cfg.linear_num_key_heads, cfg.linear_num_value_heads, cfg.linear_key_head_dim, \
            cfg.linear_value_head_dim
        C = cfg.conv_dim
        gdn_in = gdn_proj_width(cfg)       # row stride of the GDN projection (zero-padded weight rows)
        att_in = hq * 2 * D + 2 * hkv * D
        VD = cfg.value_dim
        I = cfg.intermediate_size

        ids_d = torch.tensor(list(ids), dtype=torch.long, device=dev)
        # positions 0 .. T - 1, then the sequence as one packed row: its slot and offset (0) and its length
        index = torch.arange(T + 1, dtype=torch.long, device=dev)
        pos, row0, row_len = index.data_ptr(), index.data_ptr(), index[T:].data_ptr()
        # one buffer per role of an activation, reused by every layer
        hidden, normed, mix = (torch.empty(T, H, dtype=bf16, device=dev) for _ in range(3))
        proj = torch.empty(T * max(gdn_in, att_in, 2 * I), dtype=bf16, device=dev)
        mid = torch.empty(T * max(C, hq * D, I), dtype=bf16, device=dev)
        heads = torch.empty(T * max(2 * VD, (hq + hkv) * D), dtype=bf16, device=dev)
        proj_p, mid_p, heads_p, normed_p, mix_p = (t.data_ptr() for t in (proj, mid, heads, normed, mix))
        gdn_proj, att_proj, gate_up = (proj[:T * n].view(T, n) for n in (gdn_in, att_in, 2 * I))
        gated, att, act = heads[T * VD:2 * T * VD].view(T, VD), mid[:T * hq * D].view(T, hq * D), mid[:T * I].view(T, I)
        n_gdn = sum(1 for k, _ in self.kind if k == "linear_attention")
        state = torch.zeros(n_gdn, hv, kd, vd, dtype=torch.float32, device=dev)
        ws_bytes = max(int(lib().hsg_gdn_chunk_segment_workspace_bytes(1, T, hv)), 256) if n_gdn else 256
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        mm = torch.mm
        check(L.hsg_embed_rmsnorm(ids_d.data_ptr(), self.emb.data_ptr(), cfg.vocab_size,
                                  self.layers[0]["in_w1"].data_ptr(), eps, hidden.data_ptr(), normed_p, T, H, st),
              "hsg_embed_rmsnorm")
        for i, ((kind, idx), Lw) in enumerate(zip(self.kind, self.layers)):
            if kind == "linear_attention":
                mm(normed, Lw["w_in"].t(), out=gdn_proj)
                check(L.hsg_conv_silu_update(proj_p, gdn_in, None, 0, Lw["conv_w"].data_ptr(),
                                             cfg.linear_conv_kernel_dim, None, row_len, row0, 1, T, C, mid_p, C, st),
                      "hsg_conv_silu_update")
                check(L.hsg_gdn_chunk_prefill(
                    mid_p, C, 0, cfg.key_dim, 2 * cfg.key_dim, proj_p + 2 * (C + VD + hv), proj_p + 2 * (C + VD), gdn_in,
                    Lw["A_log"].data_ptr(), Lw["dt_bias"].data_ptr(), state[idx].data_ptr(), 0, 1, row0,
                    row_len, row0, 1, T, nh, hv, kd, vd, kd ** -0.5, heads_p, None, 0, ws.data_ptr(), ws_bytes, st),
                      "hsg_gdn_chunk_prefill")
                check(L.hsg_gated_rmsnorm(heads_p, VD, proj_p + 2 * C, gdn_in, Lw["norm_w"].data_ptr(), eps,
                                          heads_p + 2 * T * VD, VD, T, hv, vd, st), "hsg_gated_rmsnorm")
                mm(gated, Lw["w_out"].t(), out=mix)
            else:
                mm(normed, Lw["w_in"].t(), out=att_proj)
                k_p = heads_p + 2 * T * hq * D
                check(L.hsg_norm_rope(proj_p, att_in, 2 * D, hq, Lw["q_w1"].data_ptr(), eps, heads_p, hq * D, D,
                                      proj_p + 2 * hq * 2 * D, att_in, D, hkv, Lw["k_w1"].data_ptr(), eps, k_p,
                                      hkv * D, D, pos, self.inv_freq.data_ptr(), cfg.rotary_dim, T, D, st),
                      "hsg_norm_rope")
                for first in range(0, T, SEG * MAX_ATT_SEGMENTS):
                    check(L.hsg_window_attention(
                        heads_p, hq * D, G * D, D, k_p, hkv * D, D, proj_p + 2 * (hq * 2 * D + hkv * D), att_in, D,
                        proj_p, att_in, G * 2 * D, 2 * D, D, row_len, row0, 1, T, first, SEG * MAX_ATT_SEGMENTS, W,
                        hkv, G, D, D ** -0.5, mid_p, hq * D, G * D, D, st), "hsg_window_attention")
                mm(att, Lw["w_out"].t(), out=mix)
            check(L.hsg_add_rmsnorm(hidden.data_ptr(), mix_p, Lw["post_w1"].data_ptr(), eps, normed_p, T, H, st),
                  "hsg_add_rmsnorm")
            mm(normed, Lw["w_gu"].t(), out=gate_up)
            check(L.hsg_silu_mul(proj_p, 2 * I, I, mid_p, T, st), "hsg_silu_mul")
            mm(act, Lw["w_down"].t(), out=mix)
            nxt = self.layers[i + 1]["in_w1"] if i + 1 < len(self.layers) else self.final_w1
            check(L.hsg_add_rmsnorm(hidden.data_ptr(), mix_p, nxt.data_ptr(), eps, normed_p, T, H, st),
                  "hsg_add_rmsnorm")
        R, E = len(self.roles), cfg.head_hidden
        h32 = self.head32
        y = torch.addmm(h32["b1"], normed.float(), h32["w1"].t())
        probs = torch.empty(R, T, 3, dtype=torch.float32, device=dev)
        check(L.hsg_risk_head_f32(y.data_ptr(), R * E, h32["ln_w"].data_ptr(), h32["ln_b"].data_ptr(),
                                  h32["w2"].data_ptr(), h32["b2"].data_ptr(), cfg.layer_norm_eps, R, E,
                                  probs.data_ptr(), T, st), "hsg_risk_head_f32")
        return probs
