"""Key norm / rotation and the paged store of long steps, by wavefronts and, from 192 tiles of 64 tokens of a head on (32-bit: 320), by tiles: whole and ragged last tiles, head sizes that
fill no power of two of lanes, tokens without a slot, slots in any order, against the definition in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.bfloat16, 2.0 ** -8)], ids=["f32", "bf16"])
@pytest.mark.parametrize("n,G,d,dv,rot,norm", [(2048, 2, 64, 64, 0, True), (2049, 1, 128, 256, 128, True), (2111, 3, 72, 40, 20, False),
                                               (4095, 2, 256, 8, 6, True), (2175, 4, 8, 128, 8, False),
                                               (6145, 2, 64, 64, 0, True), (3073, 8, 128, 256, 128, True), (2111, 6, 72, 40, 20, False),
                                               (2111, 8, 256, 8, 6, True), (2175, 6, 8, 128, 8, False), (2048, 6, 64, 64, 64, True),
                                               (6833, 3, 72, 40, 20, False), (2049, 10, 8, 128, 8, True)])
def test_stored_keys_and_values(n, G, d, dv, rot, norm, dtype, tol):
    from nano_vllm_amd import ops_seq
    g = torch.Generator().manual_seed(n + d)
    block = 16
    pages = n // block + 9
    proj = torch.randn(n, G * (d + dv) + 24, generator=g).to(dtype)
    k, v = proj[:, 8:8 + G * d], proj[:, 8 + G * d:8 + G * (d + dv)]
    w = (1 + torch.randn(d, generator=g)).to(dtype) if norm else None
    slots = torch.randperm(pages * block, generator=g)[:n].int()
    slots[[0, 63, 64, n - 1]] = -1
    pos = torch.randint(0, 5000, (n,), generator=g)
    freq = torch.rand(rot // 2, generator=g) if rot else None
    dev = proj.cuda()
    kc = torch.full((pages * block, G, d), 7.0, dtype=dtype, device="cuda")
    vc = torch.full((pages * block, G, dv), 7.0, dtype=dtype, device="cuda")
    ops_seq.knorm_kvstore(dev[:, 8:8 + G * d], dev[:, 8 + G * d:8 + G * (d + dv)], None if w is None else w.cuda(), 1e-5, G, d, dv, block,
                          slots.cuda(), kc, vc, pos.cuda() if rot else None, freq.cuda() if rot else None)
    want = k.double().view(n, G, d)
    if norm:
        want = want / torch.sqrt(want.pow(2).mean(2, keepdim=True) + 1e-5) * w.double()
    if rot:
        turn = (pos.float()[:, None] * freq).double()           # the angle is a 32-bit product
        a, b = want[..., 0:rot:2].clone(), want[..., 1:rot:2].clone()
        want = want.clone()
        want[..., 0:rot:2] = a * turn.cos()[:, None] - b * turn.sin()[:, None]
        want[..., 1:rot:2] = b * turn.cos()[:, None] + a * turn.sin()[:, None]
    kept = slots >= 0
    at = slots[kept].long()
    kc, vc = kc.cpu(), vc.cpu().view(pages, G, dv, block).permute(0, 3, 1, 2).reshape(pages * block, G, dv)
    # a stored entry is one rounding of a 32-bit value (tol x its size; a turned pair mixes two entries)
    size = want[kept].abs().amax(2, keepdim=True)
    assert ((kc[at].double() - want[kept]).abs() <= tol * size).all()
    assert torch.equal(vc[at], v[kept].view(-1, G, dv))
    rest = torch.ones(pages * block, dtype=torch.bool)
    rest[at] = False
    assert (kc[rest] == 7).all() and (vc[rest] == 7).all()
