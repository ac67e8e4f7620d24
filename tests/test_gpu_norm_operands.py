"""The norm's pass that also writes the prefill kernels' fp16 operand (csrc/e2e_glue.hip): kr_rmsnorm_q4_mlp gives the
bits of kr_rmsnorm and kr_q4_mlp, whose conversion is a launch of its own, at the edges of the rule: the fewest rows of
the prefill operands, one to four pieces per thread (the last partly filled), and rows too long for one pass.
"""
import pytest
import torch

from _util import dev_bf16, host_bits, q4_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,hidden,inter", [(64, 128, 128), (65, 2048, 256), (131, 2112, 192), (70, 4160, 128),
                                            (66, 8192, 128), (66, 8256, 128)])
def test_norm_writes_operand_bitwise(kq, m, hidden, inter):
    from kriya_q4 import synth
    print(f"[case] norm with operand m={m} hidden={hidden} inter={inter}", flush=True)
    G, U, D = (q4_dev(kq, synth.q4_weight(n, k, 6100 + i))
               for i, (n, k) in enumerate(((inter, hidden), (inter, hidden), (hidden, inter))))
    ln = dev_bf16(synth.bf16_normal((1, hidden), 6110))[0].contiguous()
    h0 = dev_bf16(synth.bf16_normal((m, hidden), 6111))
    h0[3] *= 0.0
    ln[:2] *= 1e6  # beyond fp16's range: the operand holds infinities, the tiles fall back to x
    want, got = h0.clone(), h0.clone()
    kq.mlp(G, U, D, want, x=kq.rmsnorm(want, ln, 1e-6))
    kq.rmsnorm_mlp(G, U, D, got, ln, 1e-6)
    torch.cuda.synchronize()
    assert (host_bits(got) == host_bits(want)).all()
