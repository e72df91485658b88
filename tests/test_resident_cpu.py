"""Host side of the resident loops' memory: what a full-storage FWI group leaves for the ring of the receiver
pass (fwi.resident_ring_bytes)."""
import torch

from elastic_isotropic_operators_amd.fwi import ElasticFwi, resident_ring_bytes


def test_resident_ring_bytes():
    n = 600 * 1592
    assert resident_ring_bytes(32, 600, 1592, 3000, 4) == 33 * 5 * 4 * n     # one shot on the chip
    assert resident_ring_bytes(8, 280, 472, 1000, 4) == 33 * 5 * 4 * 280 * 472 * 6   # 40 tiles a shot
    assert resident_ring_bytes(8, 280, 472, 20, 8) == 20 * 5 * 8 * 280 * 472 * 3
    assert resident_ring_bytes(4, 1028, 3028, 1000, 4) == 0                  # does not fit: launched
    for nz, nx, size in [(17, 40, 4), (72, 72, 4), (72, 40, 8), (600, 1592, 4), (1032, 1032, 4), (280, 472, 8), (9, 40000, 8)]:
        assert resident_ring_bytes(10 ** 6, nz, nx, 10 ** 4, size) < 1.1e9


def test_full_storage_group_leaves_room_for_the_ring(monkeypatch):
    """A group that is sized to the free memory keeps the ring's share of it free."""
    e = ElasticFwi.__new__(ElasticFwi)
    e.device, e.dtype = torch.device("cpu"), torch.float32
    e.nz, e.nx, e.nts, e.nshot = 280, 472, 100, 64
    ring = resident_ring_bytes(e.nshot, e.nz, e.nx, e.nts, 4)
    per_shot = (2 * e.nts + 60) * e.nz * e.nx * 4
    for free in (0, ring // 2, ring, ring + per_shot, 10 * ring):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d, f=free: (f, f))
        g = e.full_storage_group(margin=1.0)
        assert g >= 0 and (g == 0 or g * per_shot + ring <= free < (g + 1) * per_shot + ring)
