"""Every layout and epilogue of an fp16 GEMM whose plan has 256-row tiles, with a partial last row of tiles: digests of the outputs, each compared
with an fp32 product first.  As a program (the library reads LG_GEMM_TILE_WIDTH once per process) it prints them as JSON."""
import hashlib
import importlib
import json

import torch

M, N, K, S, D = 1000, 12288, 192, 250, 128     # 4 x 64 tiles of 256 x 192


def outputs():
    capi = importlib.import_module("24ppopp-liger_amd.capi")
    stream = torch.cuda.current_stream().cuda_stream
    capi.check(capi.lib.lg_stream_attach(stream, 0), "lg_stream_attach")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    draw = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)
    X, W, bias = draw(M, K).half(), (0.05 * draw(K, N)).half(), (0.3 * draw(N)).half()
    y = X.float() @ W.float()
    yb = y.half().float() + bias.float()
    gelu = lambda v: 0.5 * v * (1.0 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v * v * v)))
    idx = torch.arange(N, device="cuda")
    idx = (idx // 32) * 16 + idx % 16 + torch.where(idx % 32 >= 16, N // 2, 0)      # (gate, up) in blocks of 16
    Wg, bg = W[:, idx].contiguous(), bias[idx].contiguous()
    digests = {}
    for layout in (0, 1, 2):

        def weight(w):
            if layout == 0:
                return w, N
            t = w.t().contiguous()
            if layout == 1:
                return t, K
            blocks = torch.empty_like(t)
            capi.call("lg_weight_tile_f16", blocks.data_ptr(), t.data_ptr(), N, K, 1, K, stream)
            return blocks, K

        (w, ld), (wg, _) = weight(W), weight(Wg)
        for name, epi, rows, ref in (("plain", 0, N, y), ("bias", 1, N, yb), ("gelu", 2, N, gelu(yb)),
                                     ("heads", 3, S, yb.view(M // S, S, N // D, D).transpose(1, 2).reshape(M, N)),
                                     ("geglu", 5, N // 2, gelu(yb[:, :N // 2]) * yb[:, N // 2:])):
            out = torch.empty(ref.shape, device="cuda", dtype=torch.float16)
            b = bg if epi == 5 else bias
            heads = (S, D, N // D) if epi == 3 else (0, 0, 0)
            capi.call("lg_gemm_fused_f16", layout, N, M, K, (wg if epi == 5 else w).data_ptr(), ld, X.data_ptr(), K, out.data_ptr(), rows, epi,
                      b.data_ptr() if epi else None, *heads, stream)
            torch.cuda.synchronize()
            err = float((out.float() - ref).abs().max() / ref.abs().max())
            assert err < 4e-3, (layout, name, err)
            digests["%d %s" % (layout, name)] = hashlib.sha256(out.cpu().numpy().tobytes()).hexdigest()
    return digests


if __name__ == "__main__":
    print(json.dumps(outputs()), flush=True)
