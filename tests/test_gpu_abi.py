"""GPU: design libraries of older ABIs. A descriptor that ends where ABI 8 or 9
ended (what follows it in memory is garbage) runs with the kernels it has: no
helped kernel, no bit-plane plans, the same hashes."""
import ctypes as C

import pytest

import abi_offsets
import oracle
from rtlflow_amd.designs import registry
from rtlflow_amd.model import MODE_BITPLANE, MODE_FUSED, Model

SEED = registry.SEED_CFG[2]


@pytest.mark.gpu
@pytest.mark.parametrize("abi,size", [(8, abi_offsets.ABI9), (9, abi_offsets.ABI10)])
@pytest.mark.parametrize("name,mode", [("net_small", MODE_BITPLANE), ("net_ram", MODE_BITPLANE), ("alu", MODE_FUSED)])
def test_older_descriptors_run(gpu, abi, size, name, mode):
    lib = registry.get(name).load()
    own = lib.desc
    raw = bytearray(C.string_at(own, size)) + bytearray(b"\xff" * 256)
    raw[0:4] = abi.to_bytes(4, "little")
    old = C.create_string_buffer(bytes(raw), len(raw))
    hashes = []
    try:
        for desc in (own, C.addressof(old)):
            lib.desc = desc
            with Model(lib, 200) as m:
                m.begin(SEED)
                m.run_cycles(23, mode)
                hashes.append(m.hashes())
    finally:
        lib.desc = own
    assert (hashes[0] == hashes[1]).all()
    if mode == MODE_BITPLANE:
        want = oracle.netlist_run(registry.table_bytes(name), SEED, nstim=200, cycles=23)
        assert (hashes[1] == want).all()
