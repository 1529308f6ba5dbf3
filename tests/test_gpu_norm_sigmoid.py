"""The gate's sigmoid is the same fp32 number whatever the type of the data: 2-byte data rounds the result, not the way to it."""
import pytest
import torch

from hdla_hip.normalize import normalize_fn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [0, 1])                      # every second of the values, so that a row is one group in registers
def test_sigmoid_of_two_byte_data_is_that_of_fp32_data(first):
    """One row with x = do = 1 and an eps beside which the mean square vanishes: sigma is 2^20, c makes up for it, and the weight's
    gradient, fp32 for either type of data, is the sigmoid itself.  All gates of 2-byte type from 2^-6 to 256, both signs: beyond
    -87.3 the sigmoid is subnormal, beyond -88.7 its exponential overflows."""
    half = torch.arange(0x3c80, 0x4381, dtype=torch.int32)[first::2].to(torch.int16).view(torch.bfloat16)
    gate = torch.cat([half, -half])
    E = (gate.numel() + 7) // 8 * 8
    gate = torch.cat([gate, gate[:E - gate.numel()]]).cuda()
    got = []
    for dtype in (torch.bfloat16, torch.float32):
        x = torch.ones(1, E, dtype=dtype, device="cuda")
        w = torch.ones(E, device="cuda", requires_grad=True)
        # o = c / sqrt(E) x' / sigma w with sigma = sqrt(sum x'^2 / E + 2^40) = 2^20
        o = normalize_fn(x, w, gate=gate.to(dtype)[None], gate_pos="pre", c=float(torch.tensor(float(E)).sqrt()) * 2 ** 20, eps=2.0 ** 40)
        got.append(torch.autograd.grad(o, w, torch.ones_like(o))[0])
    exact = torch.sigmoid(gate.double())
    scale = got[1].double() @ exact / (exact @ exact)          # c / sqrt(E) / 2^20: 1 up to its rounding
    assert abs(float(scale) - 1) < 1e-6
    # exponential: the argument times log2 e (|x| 2^-24 for the product's rounding, under a quarter of that for the constant's), two
    # units of the instruction; sum, quotient and product half a unit each, the scale measured here another
    normal = gate > -70                                        # (below, the quotient by sigma is subnormal on the way)
    err = (got[1].double() / scale / exact - 1).abs()[normal]
    bound = ((1.25 * gate.double().abs() + 6) * 2.0 ** -24)[normal]
    print("largest share of the bound", float((err / bound).max()), flush=True)
    assert bool((err <= bound).all())
    assert bool((got[1][~normal].double() <= 2.0 ** -100).all())
    assert torch.equal(got[0], got[1])
