"""What the C entry points launch, on a host without a GPU: run as a program with the shim's path and the name of a
scenario below, it loads libjqmc_hip.so over the recording HIP shim (hip_host_shim.c) and prints the scenario's
result as JSON.  Device pointers are made up; nothing reads them."""

import ctypes
import json
import os
import re
import sys

FAKE = ctypes.c_void_p(0x10000)


class Host:
    def __init__(self, shim):
        self.shim = ctypes.CDLL(shim, mode=ctypes.RTLD_GLOBAL)  # before anything that needs the real runtime
        self.shim.shim_record.restype = ctypes.c_char_p
        sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
        from jqmc_amd import _lib

        self.lib = _lib

    def pack(self, ham, **kw):
        from jqmc_amd._pack import SystemPack

        return SystemPack(ham, **kw)

    def walkers(self):
        w = self.lib.Walkers()
        for name, _ in self.lib.Walkers._fields_:
            setattr(w, name, FAKE.value)
        return w

    def bytes(self, fn, pack, W):
        n = ctypes.c_int64()
        self.lib.call(fn, pack.handle, W, ctypes.byref(n))
        return n.value

    def launches(self, fn, *args):
        """The launches of one call as (kernel, grid x, grid y, block, dynamic LDS, device, refused); raises if the
        call does."""
        self.shim.shim_clear()
        self.lib.call(fn, *args)
        out = []
        for i in range(self.shim.shim_count()):
            f = self.shim.shim_record(i).decode().split()
            name = re.match(r"_ZN4jqmc(\d+)(.*)", f[0])
            out.append([name.group(2)[: int(name.group(1))] if name else f[0], *(int(f[k]) for k in (1, 2, 4, 5, 6, 7))])
        return out

    def local_energy(self, pack, W):
        n = self.bytes("jqmc_local_energy_workspace_bytes", pack, W)
        return self.launches("jqmc_local_energy", pack.handle, W, ctypes.byref(self.walkers()), None, FAKE, None, None,
                             None, FAKE, n, None)

    def position_grads(self, pack, W):
        n = self.bytes("jqmc_position_grads_workspace_bytes", pack, W)
        return self.launches("jqmc_position_grads", pack.handle, W, ctypes.byref(self.walkers()), None, 1, FAKE, FAKE,
                             FAKE, FAKE, FAKE, FAKE, FAKE, FAKE, n, None)


def large_lds(host):
    """Systems on two devices: local energy and forces of a 28-orbital system (more than 64 KiB of LDS a block)."""
    from jqmc_amd import synthetic

    ham = synthetic.chain_ecp(56, 1).hamiltonian_data
    out = []
    for dev in (0, 1):
        host.shim.shim_set_device(dev)
        for prec in ("fp64", "mixed"):
            pack = host.pack(ham, precision=prec)
            out += host.local_energy(pack, 100)
            if prec == "fp64":
                out += host.position_grads(pack, 100)
    return out


def many_walkers(host):
    """H2 with the most walkers that the set-up takes in one launch: set-up, local energy, one projection and the
    parameter derivatives."""
    from jqmc_amd import synthetic

    st = synthetic._structure(["H", "H"], [[0.0, 0.0, 0.0], [0.0, 0.0, 1.4]])
    pack = host.pack(synthetic._assemble("h2", st, {"H": "1s"}, 1, use_j3=False).hamiltonian_data)
    W = (1 << 25) - 8
    p = ctypes.byref(host.walkers())
    out = host.launches("jqmc_walkers_init", pack.handle, W, p, FAKE, 1 << 60, None)
    out += host.local_energy(pack, W)
    prm = host.lib.LrdmcParams(mode=0, n_steps=1, alat=0.3, E_scf=0.0, tau=0.0, non_local_move=0, random_mesh=1)
    out += host.launches("jqmc_lrdmc_projection", pack.handle, W, p, ctypes.byref(prm), 1, 0, FAKE, FAKE, FAKE, FAKE,
                         FAKE, FAKE, FAKE, 1 << 60, None)
    out += host.launches("jqmc_dln_psi_dparams", pack.handle, W, p, 15, FAKE, 1 << 10, FAKE, 1 << 60, None)
    return out


def long_forces(host):
    """Forces of the most water walkers that are taken at once, and of one more: electrons per launch of the
    kinetic kernel, and the workspaces of both calls."""
    from jqmc_amd import synthetic

    pack = host.pack(synthetic.water_ae(0).hamiltonian_data)
    most = (1 << 17) // 10
    return [[[r[1] for r in host.position_grads(pack, W) if r[0] == "k_fr_kinetic"],
             host.bytes("jqmc_position_grads_workspace_bytes", pack, W)] for W in (most, most + 1)]


if __name__ == "__main__":
    print(json.dumps(globals()[sys.argv[2]](Host(sys.argv[1]))))
