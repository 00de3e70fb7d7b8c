"""Netlists that the gate-net engine's LDS form runs in each of its kernel
instances: planes of 1, 2 or 4 bytes, batches of 1 or 4 wavefront rows; and one
with more RAMs than the 14 wavefronts that serve them. test_gnplan.py asserts
the instance of each, test_gpu_gatenet.py runs them."""
import numpy as np

from rtlflow_amd.designs.netlist import MUX, generate

# name: (plane bytes, wavefront rows of a batch, generator's arguments, levels
# of a multiplexer chain put behind the first output: the deeper the netlist,
# the fewer rows a level has)
NETS = {
    "u32 batches of 1": (4, 1, dict(n_gates=900, n_ff=90, n_pi=100, n_po=40, depth=9, n_rams=2, ram_depth=48,
                                    ram_width=20), 0),
    "u32 batches of 4": (4, 4, dict(n_gates=60000, n_ff=6000, n_pi=128, n_po=64, depth=5, n_rams=1, ram_depth=16,
                                    ram_width=64), 0),
    "u16 batches of 1": (2, 1, dict(n_gates=120000, n_ff=40000, n_pi=128, n_po=64, depth=8), 100),
    "u16 batches of 4": (2, 4, dict(n_gates=120000, n_ff=40000, n_pi=128, n_po=33, depth=8, n_rams=2, ram_depth=64,
                                    ram_width=33), 0),
    "u8 batches of 1": (1, 1, dict(n_gates=180000, n_ff=75000, n_pi=65, n_po=17, depth=30), 150),
    "u8 batches of 4": (1, 4, dict(n_gates=180000, n_ff=75000, n_pi=64, n_po=9, depth=30, n_rams=1, ram_depth=100,
                                   ram_width=7), 0),
    "20 RAMs": (4, 1, dict(n_gates=9000, n_ff=900, n_pi=64, n_po=64, depth=9, n_rams=20, ram_depth=32, ram_width=8), 0),
}
LDS_BYTES = 160 * 1024 - 64


def table(name: str):
    kw, chain = NETS[name][2:]
    t = generate(seed=0x99, **kw)[1]
    if chain:
        rng = np.random.default_rng(chain)
        n0 = t.first_gate + t.n_gates
        gin = rng.integers(0, n0, (chain, 3)).astype(np.uint32)
        gin[:, 1 + rng.integers(0, 2)] = np.concatenate([[t.po[0]], n0 + np.arange(chain - 1)])
        t.gate_type = np.concatenate([t.gate_type, np.full(chain, MUX, np.uint8)])
        t.gate_in = np.concatenate([t.gate_in, gin])
        t.po[0] = n0 + chain - 1
    return t
