"""The scalar offsets of the small tiles' memory requests, from the built code objects, on the CPU.

A buffer request's range check compares the lane's offset with the resource's length minus the request's scalar offset.
That difference may not wrap: a scalar offset past the length (a negative one among them) would let lanes through that
the length was to stop, and the small tiles stop whole requests by a length of zero (the steps before their first k
group). Here each wave's scalar instructions are stepped through on the host, with made-up operand addresses, and every
buffer request must have a scalar offset from 0 to its resource's length. Values that come from lanes are unknown
(a branch on the lanes' mask falls through); a request's scalar operands must be known.
"""
import re
import struct

import pytest

from tests.test_ring_schedule import _disassembly

M32, M64 = (1 << 32) - 1, (1 << 64) - 1


def _s32(v):
    return v - (1 << 32) if v >> 31 else v


def _f32(v):
    return struct.unpack("<f", struct.pack("<I", v & M32))[0]


def _bits(x):
    return struct.unpack("<I", struct.pack("<f", x))[0]


class Wave:
    """The scalar state of one wave: registers by number (vcc apart), scc, and the vector registers that hold
    one known value in all lanes."""

    def __init__(self, kernarg, workgroup, wave):
        self.kernarg, self.vcc, self.scc, self.requests = kernarg, None, 0, []
        self.s = {0: 0x100000, 1: 0, 2: workgroup[0], 3: workgroup[1]}
        self.v, self.tid0 = {}, 64 * wave

    def regs(self, t):  # "s7" -> (7, 1), "s[4:7]" -> (4, 4)
        a, _, b = t[1:].strip("[]").partition(":")
        return int(a), int(b or a) - int(a) + 1

    def get(self, t, wide=False):
        if t == "vcc":
            return self.vcc
        if t == "exec":
            return M64
        if t[0] == "s":
            a, n = self.regs(t)
            r = [self.s.get(a + i) for i in range(2 if wide else 1)]
            return None if None in r else sum(x << (32 * i) for i, x in enumerate(r))
        return int(t, 0) & (M64 if wide else M32)

    def put(self, t, v, wide=False):
        if t == "vcc":
            self.vcc = v
        elif t[0] == "s" and t[1] in "[0123456789":
            a, _ = self.regs(t)
            for i in range(2 if wide else 1):
                self.s[a + i] = None if v is None else (v >> (32 * i)) & M32

    def load(self, t, base, off):
        a, n = self.regs(t)
        at = self.get(base, True) - 0x100000 + int(off, 0)
        for i in range(n):
            self.s[a + i] = struct.unpack_from("<I", self.kernarg, at + 4 * i)[0]

    def alu(self, op, d, *src):
        """A two- or one-operand scalar instruction."""
        name, _, ty = op[2:].rpartition("_")
        wide = ty == "b64"
        a, *r = [self.get(t, wide) for t in src]
        b = r[0] if r else 0
        if name == "cselect":
            assert self.scc is not None, op
            return self.put(d, a if self.scc else b, wide)
        if name in ("addk", "mulk", "movk"):  # d op= immediate
            name, a, b = name[:-1], a if name == "movk" else self.get(d), a
        if a is None or b is None:
            self.scc = None if name not in ("mov", "mul", "mul_hi") else self.scc
            return self.put(d, None, wide)
        top = M64 if wide else M32
        sa, sb = (_s32(a), _s32(b)) if not wide else (a, b)
        carry = self.scc if name == "addc" else 0
        v = {"mov": a, "add": a + b, "addc": a + b + (carry or 0), "sub": a - b, "mul": a * b, "and": a & b, "or": a | b,
             "xor": a ^ b, "andn2": a & ~b, "lshl": a << (b & (63 if wide else 31)), "lshr": a >> (b & 31),
             "ashr": sa >> (b & 31), "abs": abs(sa),
             "mul_hi": (a * b if ty == "u32" else sa * sb) >> 32,
             "min": min(a, b) if ty == "u32" else min(sa, sb) & M32,
             "max": max(a, b) if ty == "u32" else max(sa, sb) & M32}[name]
        self.put(d, v & top, wide)
        if name in ("add", "addc"):
            self.scc = int(v > M32) if ty == "u32" else None
        elif name in ("min", "max"):
            self.scc = int(v & top == a)
        elif name not in ("mov", "mul", "mul_hi"):
            self.scc = int(v & top != 0) if name != "sub" else None

    def cmp(self, op, x, y):
        _, _, rel, ty = op.split("_")
        a, b = self.get(x, ty == "u64"), self.get(y, ty == "u64")
        assert a is not None and b is not None, op
        if ty == "i32":
            a, b = _s32(a), _s32(b)
        self.scc = int({"lt": a < b, "le": a <= b, "gt": a > b, "ge": a >= b, "eq": a == b, "lg": a != b}[rel])

    def valu(self, op, args):
        """The vector instructions that wave-uniform values pass through; the others' results are unknown."""
        def val(t):
            return self.v.get(int(t[1:])) if t[0] == "v" and t != "vcc" else self.get(t)

        name = re.sub("_e(32|64)$", "", op)
        if name == "v_readfirstlane_b32":
            return self.put(args[0], self.tid0 if args[1] == "v0" else val(args[1]))
        f = {"v_cvt_f32_u32": lambda a: _bits(float(a)), "v_rcp_iflag_f32": lambda a: _bits(1.0 / _f32(a)),
             "v_mul_f32": lambda a, b: _bits(_f32(a) * _f32(b)), "v_cvt_u32_f32": lambda a: int(_f32(a)),
             "v_mov_b32": lambda a: a, "v_max_i32": lambda a, b: max(_s32(a), _s32(b)), "v_add_u32": lambda a, b: a + b,
             "v_min_i32": lambda a, b: min(_s32(a), _s32(b)), "v_sub_u32": lambda a, b: a - b,
             "v_subrev_u32": lambda a, b: b - a, "v_sub_co_u32": lambda a, b: a - b}.get(name)
        dst = 2 if name.endswith("_co_u32") or name.startswith("v_mad_") else 1
        a = [val(t) for t in args[dst:]] if f else [None]
        v = None if None in a else f(*a)
        for t in args[:dst]:
            if t == "vcc" or t[0] == "s":  # a lane mask: here a borrow, equal in all lanes
                self.put(t, None if v is None else M64 if v < 0 else 0, True)
            else:
                r, n = self.regs(t)
                for i in range(n):
                    self.v[r + i] = None if v is None else v & M32

    def run(self, ins, limit=200000):
        at = {a: i for i, (a, _, _) in enumerate(ins)}
        i = 0
        for _ in range(limit):
            a, op, arg = ins[i]
            args = [t.strip() for t in arg.split("<")[0].split(",")]
            i += 1
            if op == "s_endpgm":
                return self.requests
            if op.startswith(("s_branch", "s_cbranch")):
                k = int(args[0])
                taken = {"s_branch": 1, "s_cbranch_scc1": self.scc, "s_cbranch_execz": 0, "s_cbranch_vccnz": self.vcc,
                         "s_cbranch_vccz": None if self.vcc is None else self.vcc == 0,
                         "s_cbranch_scc0": None if self.scc is None else not self.scc}[op]
                assert taken is not None, f"{op} at {a:#x} on an unknown value"
                if taken:
                    i = at[a + 4 + 4 * (k - 65536 if k >> 15 else k)]
            elif op.startswith("s_load"):
                self.load(*args)
            elif op.startswith("s_cmp"):
                self.cmp(op, *args)
            elif op.startswith(("buffer_load", "buffer_store")):
                srsrc, soff = [t for t in args if t.startswith("s[")][0], arg.split(" offen")[0].split(",")[-1].strip()
                r, _ = self.regs(srsrc)
                self.requests.append((a, self.get(soff), self.s.get(r + 2)))
            elif op.startswith("v_"):
                self.valu(op, args)
            elif op.startswith("s_and_saveexec"):
                self.put(args[0], None, True)
                self.scc = None
            elif op.startswith("s_") and not op.startswith(("s_nop", "s_waitcnt", "s_barrier")):
                self.alu(op, *args)
        raise AssertionError("no end within the limit")


TILES = [("16x32", 2, 8), ("16x64", 4, 8), ("16x128", 8, 4), ("32x128", 8, 4), ("48x128", 8, 4), ("80x128", 8, 3),
         ("32x256", 8, 3), ("48x256", 8, 3), ("64x256", 8, 3)]  # tile, waves, stages


@pytest.mark.parametrize("out", ["bf16", "e4m3"])
@pytest.mark.parametrize("tile,waves,stages", TILES)
def test_scalar_offsets_stay_within_the_resources(out, tile, waves, stages):
    """Every remainder of the k groups by the stages, the first and the last tile, first and last wave. The requests of
    the steps before the first k group (5 or 10 of weights a wave, and the activations') have length 0."""
    rows, weights = map(int, tile.split("x"))
    ins = _disassembly(f"kern_mx_gemm_{out}_t{tile}")
    for groups in range(1, 2 * stages + 2):
        M, N, K = 2 * rows + 1, 3 * 256, 512 * groups
        grid = (-(-N // weights), -(-M // rows))
        ptrs = [0x200000000000 + (i << 34) for i in range(5 if out == "bf16" else 6)]
        kernarg = struct.pack(f"<{len(ptrs)}Qiii4xQ", *ptrs, M, N, K, 0) + struct.pack("<3I", *grid, 1)
        for workgroup in [(0, 0), (grid[0] - 1, grid[1] - 1)]:
            for wave in (0, waves - 1):
                req = Wave(kernarg + bytes(64), workgroup, wave).run(ins)
                early = -groups % stages
                assert sum(n == 0 for _, _, n in req) >= early * 5, (groups, workgroup, wave)
                for a, soff, n in req:
                    assert soff is not None and n is not None, hex(a)
                    assert soff <= n, (f"request at {a:#x}: scalar offset {_s32(soff)} with {n} bytes "
                                       f"(K = {K}, workgroup {workgroup}, wave {wave})")
