"""The small tiles' memory requests, from the built code objects, on the CPU: scalar offsets, and hand-counted waits.

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
        self.kernarg, self.vcc, self.scc, self.requests, self.events = kernarg, None, 0, [], []
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
        if name == "bfe":  # a field: offset and width; signed, its top bit is its sign
            width = b >> 16 & 127
            f = a >> (b & 31) & ((1 << width) - 1)
            a, b, name = f - (1 << width if ty == "i32" and width and f >> (width - 1) else 0), 0, "or"
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

    def run(self, ins, stop=None, limit=200000):
        """Steps to the end of the program, or to the first `stop` instruction; the requests as (address, scalar offset,
        resource length)."""
        at = {a: i for i, (a, _, _) in enumerate(ins)}
        i = 0
        for _ in range(limit):
            a, op, arg = ins[i]
            args = [t.strip() for t in arg.split("<")[0].split(",")]
            i += 1
            if op in ("s_endpgm", stop):
                return self.requests
            if op.startswith(("s_branch", "s_cbranch")):
                k = int(args[0])
                taken = {"s_branch": 1, "s_cbranch_scc1": self.scc, "s_cbranch_execz": 0, "s_cbranch_execnz": 1, "s_cbranch_vccnz": self.vcc,
                         "s_cbranch_vccz": None if self.vcc is None else self.vcc == 0,
                         "s_cbranch_scc0": None if self.scc is None else not self.scc}[op]
                assert taken is not None, f"{op} at {a:#x} on an unknown value"
                if taken:
                    i = at[a + 4 + 4 * (k - 65536 if k >> 15 else k)]
            elif op.startswith("s_load"):
                self.load(*args)
            elif op.startswith("s_cmp"):
                self.cmp(op, *args)
            elif op.startswith("s_bitcmp"):
                v = self.get(args[0])
                self.scc = None if v is None else int(v >> (self.get(args[1]) & 31) & 1 == int(op[8]))
            elif op == "s_waitcnt":
                for c in ("vmcnt", "lgkmcnt"):
                    if m := re.search(rf"{c}\((\d+)\)", arg):
                        self.events.append((c, int(m.group(1))))
            elif op.startswith(("ds_read", "global_")):
                self.events.append((op,))
            elif op.startswith(("buffer_load", "buffer_store")):
                self.events.append(("lds_request" if arg.endswith("lds") else op,))
                srsrc, soff = [t for t in args if t.startswith("s[")][0], arg.split(" offen")[0].split(",")[-1].strip()
                r, _ = self.regs(srsrc)
                self.requests.append((a, self.get(soff), self.s.get(r + 2)))
            elif op.startswith("v_"):
                self.valu(op, args)
            elif op.startswith("s_and_saveexec"):
                self.put(args[0], None, True)
                self.scc = None
            elif op.startswith("s_") and op not in ("s_nop", "s_barrier"):
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


def _check_mxfp8_waits(ins, tile, ktiles):
    rows, weights = map(int, tile.split("x"))
    mt, ng = rows // 16, weights // 16
    M, N, K = 2 * rows, 2 * weights, 128 * ktiles - 32
    kernarg = struct.pack("<5Q4i3I", *[0x200000000000 + (i << 34) for i in range(5)], M, N, K, N, 2, 2, 1)
    for wave in range(8):
        w = Wave(kernarg + bytes(64), (1, 1), wave)
        for a, soff, n in w.run(ins, stop="s_barrier"):
            assert soff is not None and n is not None and soff <= n, hex(a)
        steps = (ktiles - wave + 7) // 8
        out, sent, arrived, reads, unread, step = [], 0, 0, 0, False, 0
        for e in w.events:
            if e[0] == "lds_request":
                assert not unread, f"wave {wave}: a request while step {step}'s reads are outstanding"
                # a slot's refill comes after its step's reads
                assert sent // (2 * mt) < 2 or reads >= (sent // (2 * mt) - 2) * 2 * (mt + ng) + 2 * mt
                out.append(True)
                sent += 1
            elif e[0].startswith(("buffer_", "global_")):
                out.append(False)
            elif e[0] == "vmcnt":
                while len(out) > e[1]:
                    arrived += out.pop(0)
            elif e[0] == "lgkmcnt" and e[1] == 0:
                unread = False
            elif e[0].startswith("ds_read"):
                step, at = divmod(reads, 2 * (mt + ng))  # 2 mt reads of activations, then 2 ng of weights
                if at < 2 * mt:
                    assert arrived >= 2 * mt * (step + 1), f"wave {wave}: step {step} of {steps} reads ahead of its wait"
                    unread = True
                reads += 1
        assert reads == 2 * (mt + ng) * steps and sent == arrived == 2 * mt * steps


@pytest.mark.parametrize("tile", ["16x16", "16x32", "16x64", "32x64", "32x128", "48x64", "64x64"])
def test_mxfp8_tiles_wait_for_their_activations(tile):
    """A wave of kern_mx_gemm_mxfp8_t* takes every eighth k-tile and has two k-tiles of activations on their way into its
    LDS, waited for by a count that depends on the step (first, last, both, neither). Its instructions as they execute,
    up to the barrier at which the waves add their sums: when a k-tile's activations are read, the requests that brought
    them have retired; a request into a slot follows a full wait for the slot's reads; none is left in flight; and scalar
    offsets stay within the resources. With none to five k-tiles a wave; a wait that is one too large is caught."""
    ins = _disassembly(f"kern_mx_gemm_mxfp8_t{tile}")
    for ktiles in (1, 8, 9, 16, 17, 24, 25, 33, 41):
        _check_mxfp8_waits(ins, tile, ktiles)
    rows, weights = map(int, tile.split("x"))
    first = f"vmcnt({weights // 8 + rows // 8})"  # the first step's, behind it the next k-tile's requests and the weights'
    late = [(a, op, arg.replace(first, f"vmcnt({weights // 8 + rows // 8 + 1})") if op == "s_waitcnt" else arg)
            for a, op, arg in ins]
    assert late != ins
    with pytest.raises(AssertionError, match="ahead of its wait"):
        _check_mxfp8_waits(late, tile, 17)
