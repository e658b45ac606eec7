"""What an execution launches (schedule.cpp): small independent instructions share launches. The joined kernels run on the
CPU (tests/cpu_emul.py) against the oracle."""
import re

import numpy as np
import pytest

import helium_amd as ha
from helium_amd.backend import Plan
from oracle import helium_ir as oracle_ir
from oracle import numerics as nm

from cpu_emul import run_kernel
from helpers import run_tile_kernel_cpu, run_with_compiler


class Case:
    """A graph, its inputs' values in storage form and the kernels that an execution of it launches."""

    def __init__(self, seed=0):
        self.g, self.host, self.rng = ha.ir.OpGraph(), {}, np.random.default_rng(seed)

    def new(self, shape, dtype="f32"):
        i = self.g.new_input(list(shape), dtype)
        self.host[i] = nm.to_storage(self.rng.uniform(-1, 1, shape).astype(np.float32), dtype)
        return i

    def launches(self):
        self.g.optimize()
        self.plan = Plan(self.g)
        return [self.plan.launch_kernel(i) for i in range(self.plan.num_launches())]

    def check(self, kernels, entries, rel=1e-4):
        """Runs `kernels` one after the other on the CPU and compares every value that leaves the graph with the oracle's."""
        pg = self.plan.graph()
        origin = {n["id"]: n["origin"] for n in pg.nodes}
        by_id = {n["id"]: n for n in self.g.nodes}
        val, _ = oracle_ir.evaluate(self.g.nodes, self.host)
        have = {n["id"]: self.host[origin[n["id"]]] for n in pg.nodes if n["node"] == "input"}
        made = {}
        for k, entry in zip(kernels, entries):
            made.update(run_tile_kernel_cpu(k, {**have, **made}, entry))
        for node, data in made.items():
            o = origin[node]
            want = np.asarray(val[o], dtype=np.float64).reshape(-1)
            got = nm.from_storage(data, by_id[o]["dtype"], want.shape).astype(np.float64).reshape(-1)
            tol = 1e-2 if by_id[o]["dtype"] == "bf16" else rel
            assert (np.abs(got - want) <= tol * np.maximum(np.abs(want), 1.0)).all(), (o, by_id[o], got[:4], want[:4])
        return made


def updates(count, seed=0):
    """`count` independent elementwise instructions, each of a shape of its own."""
    c = Case(seed)
    for k in range(count):
        c.g.new_output(c.g.change_data_type(c.g.unary(c.new([3 + k, 5 + 7 * k]), "relu"), "bf16"))
    return c


def test_small_instructions_share_a_launch():
    c = updates(3)
    kernels = c.launches()
    assert [k.description.split("\n")[0].split(" grid")[0] for k in kernels] == ["joined members=3"], [k.description for k in kernels]
    assert len(c.check(kernels, ["joined_kernels"])) == 3
    with pytest.raises(ha.HeliumError, match="no launch 1"):
        c.plan.launch_kernel(1)


@pytest.mark.parametrize("count,members", [(8, [8]), (12, [12]), (24, [24]), (25, [24, 1]), (30, [24, 6]), (49, [24, 24, 1])])
def test_a_step_of_many_small_instructions_shares_launches(count, members):
    """However many there are, as many to a launch as one takes: such a step does not fan out over streams."""
    c = updates(count, seed=count)
    kernels = c.launches()
    assert [len(k.args) for k in kernels] == [2 * m for m in members], [k.description for k in kernels]
    assert len(c.check(kernels, ["joined_kernels" if m > 1 else "pointwise_kernel" for m in members])) == count


def test_a_group_that_takes_too_many_arguments_is_split():
    c = Case(20)
    for k in range(10):  # 20 arguments each: a launch takes 160
        total = c.new([4, 4 + k])
        for _ in range(18):
            total = c.g.binary(total, c.new([4, 4 + k]), "add")
        c.g.new_output(total)
    kernels = c.launches()
    assert [len(k.args) for k in kernels] == [160, 40], [k.description for k in kernels]
    assert len(c.check(kernels, ["joined_kernels"] * 2)) == 10


def test_a_step_of_larger_instructions_fans_out():
    """2 MB each, as many as fan out over streams (HE_OPT_STREAM_FAN_OUT): no launch list."""
    c = Case()
    for _ in range(16):
        c.g.new_output(c.g.unary(c.g.unary(c.g.new_input([512, 512], "f32"), "exp"), "relu"))
    assert c.launches() == []


@pytest.mark.parametrize("terms", [159, 160, 400])
def test_an_instruction_of_many_arguments_goes_out_alone(terms):
    """A small sum of as many tensors as a shared launch takes arguments, or more, beside instructions that share one."""
    c = Case(terms)
    total = c.new([8, 8])
    for _ in range(terms - 1):
        total = c.g.binary(total, c.new([8, 8]), "add")
    c.g.new_output(total)
    for k in range(3):
        c.g.new_output(c.g.unary(c.new([5, 3 + k]), "neg"))
    kernels = c.launches()
    members = sorted(len(k.args) for k in kernels)
    assert members == [6, terms + 1], [k.description for k in kernels]
    kernels.sort(key=lambda k: len(k.args))
    made = c.check(kernels, ["joined_kernels", "pointwise_kernel"], rel=1e-5 * terms)
    assert len(made) == 4


def reductions(count, shape, dtype, seed=0):
    """`count` column reductions (a block's part of each meets in LDS) that differ in their sizes."""
    c = Case(seed)
    for k in range(count):
        c.g.new_output(c.g.reduce(c.g.swap_dims(c.new([shape[0], shape[1], shape[2] - 8 * k], dtype), 1, 2), "mean", 1))
    return c


@pytest.mark.parametrize("count,shape,dtype", [(24, (64, 32, 2048), "bf16"), (24, (128, 32, 1024), "bf16"), (5, (64, 32, 1024), "f32")])
def test_a_joined_kernel_takes_the_lds_of_its_largest_member(count, shape, dtype):
    c = reductions(count, shape, dtype)
    kernels = c.launches()
    assert len(kernels) == 1 and len(kernels[0].args) == 2 * count, [k.description for k in kernels]
    own = [c.plan.kernel(i).source for i in range(count)]
    per_thread = max(int(re.search(r"#define NV (\d+)", s).group(1)) for s in own)
    assert all("__shared__ float col_red[TY * TX * NV]" in s for s in own)
    assert f" lds={256 * per_thread * 4}\n" in kernels[0].description and kernels[0].source.count("__shared__") == 1, kernels[0].description


def test_members_with_lds_of_their_own_share_one_buffer():
    """Column reductions of two widths, rows that meet in LDS, a sum over everything, and members without any."""
    c = Case(7)
    g = c.g
    g.new_output(g.reduce(g.swap_dims(c.new([64, 32, 2048], "bf16"), 1, 2), "mean", 1))
    g.new_output(g.reduce(g.swap_dims(c.new([33, 31, 2000]), 1, 2), "max", 1))
    g.new_output(g.reduce(c.new([9, 700]), "sum", 1))
    g.new_output(g.reduce(g.unary(c.new([4, 120]), "neg"), "sum", 2))
    g.new_output(g.unary(c.new([5, 7]), "exp"))
    kernels = c.launches()
    assert len(kernels) == 1 and kernels[0].source.count("__shared__") == 1, [k.description for k in kernels]
    for name in ("col_red", "row_red", "blk_red"):
        assert f"(&{name})" in kernels[0].source, name
    assert len(c.check(kernels, ["joined_kernels"])) == 5


def test_a_join_that_does_not_compile_leaves_its_members_a_launch_each(tmp_path):
    code = """
import helium_amd as ha
from helium_amd.backend import Plan
g = ha.ir.OpGraph()
for k in range(4):
    g.new_output(g.unary(g.new_input([3, 5 + k], "f32"), "relu"))
plan = Plan(g)
print(sorted(len(plan.launch_kernel(i).args) for i in range(plan.num_launches())))
"""
    refuses = run_with_compiler(tmp_path, 'if [ "$1" = joined_kernels ]; then printf "e\\\\021\\\\0\\\\0\\\\0\\\\0\\\\0\\\\0\\\\0no registers left"; else exec "$REAL" "$@"; fi', code)
    assert refuses.stdout.split("\n")[0] == "[2, 2, 2, 2]", refuses.stdout + refuses.stderr
    assert run_with_compiler(tmp_path, 'exec "$REAL" "$@"', code).stdout.split("\n")[0] == "[8]"


@pytest.mark.parametrize("entry,graph", [
    ("joined_kernels", "for k in range(30): g.new_output(g.unary(g.new_input([3, 5 + k], 'f32'), 'relu'))"),
    ("joined_products", "for k in range(8): g.new_output(g.matmul(g.new_input([64, 64], 'bf16'), g.new_input([64, 32 + 8 * k], 'bf16'), 'bf16_f32'))")])
def test_joins_compile_side_by_side(tmp_path, entry, graph):
    """Each of two compilations of a joined kernel waits for the other to have begun (and gives up after a while)."""
    script = f"""if [ "$1" = {entry} ]; then
mkdir -p {tmp_path}/begun; : > {tmp_path}/begun/$$
n=0; while [ $(ls {tmp_path}/begun | wc -l) -lt 2 ]; do n=$((n + 1)); if [ $n -gt 200 ]; then : > {tmp_path}/alone; break; fi; sleep 0.1; done
fi
exec "$REAL" "$@"
"""
    code = f"""
import helium_amd as ha
from helium_amd.backend import Plan
g = ha.ir.OpGraph()
{graph}
print(Plan(g).num_launches())
"""
    out = run_with_compiler(tmp_path, script, code)
    assert out.stdout.strip() == "2", out.stdout + out.stderr
    assert len(list((tmp_path / "begun").iterdir())) == 2 and not (tmp_path / "alone").exists()


def held(shape, count, dtype="f32"):
    """A graph that holds `count` values of `shape` between its launches: products that other products read."""
    c = Case()
    g, precision = c.g, "f32_f32" if dtype == "f32" else "bf16_f32"
    values = [g.matmul(g.new_input([shape[0], 64], dtype), g.new_input([64, shape[1]], dtype), precision) for _ in range(count)]
    for v in values:
        g.new_output(g.matmul(v, g.new_input([shape[1], 32], dtype), precision))
    return c


def test_intermediate_values_lie_in_blocks_of_bounded_size(monkeypatch):
    GiB = 1 << 30
    small = held((1024, 1024), 3)
    small.launches()
    assert small.plan.blocks() == [3 * 4 << 20]  # one block for everything
    medium = held((16384, 8192), 5)  # 512 MiB each: two to a block
    medium.launches()
    assert medium.plan.blocks() == [GiB, GiB, GiB // 2]
    large = held((32768, 12288), 3)  # 1.5 GiB each: a block of its own
    large.launches()
    assert large.plan.blocks() == [3 * GiB // 2] * 3
    monkeypatch.setenv("HELIUM_HIP_ARENA_BLOCK", str(8 << 20))
    cut = held((1024, 1024), 3)
    cut.launches()
    assert cut.plan.blocks() == [8 << 20, 4 << 20]


def test_results_have_storage_of_their_own():
    """Reshapes are no launches where nobody can tell, and copies where two results, or a result and an input, would share."""
    def launched(build):
        c = Case()
        for node in build(c.g, c.g.new_input([6, 10], "f32")):
            c.g.new_output(node)
        return sorted(sum(a["is_output"] for a in k.args) for k in c.launches())

    total = lambda g, x: g.reduce(x, "sum", 1)  # noqa: E731
    assert launched(lambda g, x: [g.reshape(total(g, x), [6])]) == [1]                       # a value between launches
    assert launched(lambda g, x: [g.reshape(x, [60])]) == [1]                                # an input
    assert launched(lambda g, x: [g.reshape(g.reshape(x, [60]), [10, 6])]) == [1]
    assert launched(lambda g, x: [x]) == []                                                  # the input itself
    def both(g, x):
        t = total(g, x)
        return [t, g.reshape(t, [6])]
    assert launched(both) == [1, 1]
    assert launched(lambda g, x: both(g, x)[::-1]) == [1, 1]

    def three_shapes(g, x):
        t = total(g, x)
        flat = g.reshape(t, [6])
        return [g.reshape(flat, [2, 3]), flat, g.reshape(t, [3, 2])]
    assert launched(three_shapes) == [1, 3]  # (one instruction for the shapes)


# ---- joined products -------------------------------------------------------------------------------------------------
def run_product(kernel, entry, inputs):
    """A product's launch (one of several products, the classes of a strided data gradient, or one product) on the CPU."""
    gx = int(re.search(r"grid=(\d+)", kernel.description).group(1))
    threads = int(re.search(r"threads=(\d+)", kernel.description).group(1))
    bufs = [(np.full(a["numel"], np.nan, np.float32) if a["dtype"] == "f32" else np.full(a["numel"], 0x7FC0, np.uint16), 2) if a["is_output"]
            else (inputs[a["node"]], 0) for a in kernel.args]
    outs = run_kernel(re.split(r"// ---- part \d+ of \d+\n", kernel.source)[0], entry, gx, threads, bufs)
    return dict(zip([a["node"] for a in kernel.args if a["is_output"]], outs))


def conv_backward(c, image, channels, kernel, stride):
    """A strided convolution's data and filter gradients."""
    params = {"in_channels": image[3], "out_channels": channels, "kernel_size": [kernel, kernel], "stride": [stride, stride]}
    out = oracle_ir.conv_output_size(params, image[1:3], [kernel, kernel])
    dy, w, x = c.new([image[0], *out, channels], "bf16"), c.new([channels, kernel, kernel, image[3]], "bf16"), c.new(image, "bf16")
    return [c.g.conv_backward_data(dy, w, params, list(image[1:3])), c.g.conv_backward_filter(dy, x, params)]


def linear_backward(c, rows, inner, cols, dtype, precision):
    x, w, dy = c.new([rows, inner], dtype), c.new([inner, cols], dtype), c.new([rows, cols], dtype)
    return [c.g.matmul(dy, c.g.swap_dims(w, 0, 1), precision), c.g.matmul(c.g.swap_dims(x, 0, 1), dy, precision)]


def plain_and_with_an_epilogue(c, count):
    g, outs = c.g, []
    for k in range(count):
        v = g.matmul(c.new([40 + 32 * k, 96], "bf16"), c.new([96, 48 + 8 * k], "bf16"), "bf16_f32")
        outs.append(g.change_data_type(g.unary(v, "relu"), "bf16") if k % 2 else v)
    return outs


JOINED = {
    "even_bf16": lambda c: linear_backward(c, 64, 96, 128, "bf16", "bf16_f32"),
    "ragged_bf16": lambda c: linear_backward(c, 67, 101, 35, "bf16", "bf16_f32"),
    "ragged_f32": lambda c: linear_backward(c, 33, 70, 47, "f32", "f32_f32"),
    "epilogues": lambda c: plain_and_with_an_epilogue(c, 4),
    "strided_convolution": lambda c: conv_backward(c, [1, 9, 9, 16], 16, 3, 2),
    "convolution_that_leaves_pixels": lambda c: conv_backward(c, [1, 9, 9, 8], 16, 1, 2),
    "one_row_and_one_column": lambda c: [c.g.matmul(c.new([1, 200], "bf16"), c.new([200, 40], "bf16"), "bf16_f32"),
                                         c.g.matmul(c.new([50, 200], "bf16"), c.new([200, 1], "bf16"), "bf16_f32")],
}


@pytest.mark.parametrize("name", JOINED)
def test_joined_products_are_their_members(name):
    """Products that share a launch: the bits that each makes by itself, and the oracle's values."""
    c = Case(11)
    for node in JOINED[name](c):
        c.g.new_output(node)
    kernels = c.launches()
    assert len(kernels) == 1 and kernels[0].description.startswith("joined products="), [k.description for k in kernels]
    origin = {n["id"]: n["origin"] for n in c.plan.graph().nodes}
    inputs = {n: c.host[o] for n, o in origin.items() if o in c.host}
    got = run_product(kernels[0], "joined_products", inputs)
    alone = {}
    for i in range(sum(len(instrs) for instrs, _ in c.plan.steps)):
        k = c.plan.kernel(i)
        alone.update(run_product(k, "fused_matmul_parts" if k.description.startswith("composite") else "fused_matmul", inputs))
    assert sorted(got) == sorted(alone) and len(got) >= 2
    val, desc = oracle_ir.evaluate(c.g.nodes, c.host)
    for node, data in got.items():
        assert np.array_equal(data, alone[node]), (node, kernels[0].description)
        want = np.asarray(val[origin[node]], dtype=np.float64).reshape(-1)
        have = nm.from_storage(data, desc[origin[node]][1], want.shape).astype(np.float64)
        assert np.abs(have - want).max() <= (1e-5 if "f32" in name else 2e-2) * np.abs(want).max(), (node, kernels[0].description)
