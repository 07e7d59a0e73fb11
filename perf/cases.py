"""The work users of this framework have it do, as cases that can be timed and compared.

A case is a dict of plain values.  ``listed()`` holds the fixed ones, ``draw(rng)`` gives another of the same ranges,
``prepare(case, seed)`` makes what a program has in hand before the call, ``run(state)`` is one pass through the public
entry points, ``work(case)`` is what that pass cannot do without and ``tolerance(case)`` how far another correct
implementation at the same precision may be off.

Kinds:

``step``      one train step of the U-Net as the trainer runs it: device-side ingest of the loader's float32 volume and
              int16 mask, forward under bf16 autocast, fused CE + Dice, backward, the gradients laid into the flat buffer
              that a data-parallel run reduces, clipped Adam.  Returns loss, logits and that buffer.  ``plain``: the
              modules alone are this library's; input conversion, clipping and Adam stay the trainer's torch calls.
``evaluate``  the validation forward of the same program: ingest, forward under autocast without gradients.
``conv``      the three directions of one 3x3x3 convolution through the operators.
``upconv``    the three directions of one 2x2x2 stride-2 transposed convolution through the operators.
``norm``      GroupNorm + ReLU, forward and backward, through the drop-in module.
"""

import torch

import scaffold_amd as sa

CL = torch.channels_last_3d
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GROUPS = 8


def listed():
    step = dict(kind="step", n=1, halo=False, graph=False, plain=False)
    return [
        # One depth shard of a 128-cube sample on one GPU, binary occupancy, 10 classes and background: the step the
        # benchmark quotes, captured once as a HIP graph and replayed per batch.
        dict(step, name="shard_step_graph", d=64, h=128, w=128, cin=1, classes=11, base=32, layers=4, halo=True, graph=True),
        # The reference's own network (base width 64, RGB volumes, 5 categories and background) on a whole 128-cube, eager:
        # the largest step one GPU is given.
        dict(step, name="cube_step", d=128, h=128, w=128, cin=3, classes=6, base=64, layers=4),
        # The same data one problem scale down (64-cube, one level less), eager, in a trainer that took over the modules
        # and the loss head: an ordinary development run.
        dict(step, name="scale6_step", d=64, h=64, w=64, cin=3, classes=6, base=32, layers=3, plain=True),
        # The smallest problem scale in use (32-cube): the step is launches and host work.
        dict(step, name="small_step", d=32, h=32, w=32, cin=1, classes=11, base=32, layers=2),
        # A batch of two crops of odd extents: odd planes at the lower levels, padded upsampled tensors, cut tiles.
        dict(step, name="ragged_step", n=2, d=44, h=60, w=75, cin=3, classes=6, base=32, layers=3),
        # Validation between epochs: the training program's model, forward only, a volume that is no power of two.
        dict(kind="evaluate", name="evaluate", n=1, d=96, h=80, w=112, cin=3, classes=6, base=64, layers=3),
        # The convolution the benchmark's headline is quoted on.
        dict(kind="conv", name="conv_cube", n=1, d=128, h=128, w=128, cin=32, cout=32, dtype="bf16"),
        # A deep level of the network on its own: small volume, many channels, fp16.
        dict(kind="conv", name="conv_deep", n=1, d=8, h=16, w=16, cin=256, cout=256, dtype="fp16"),
        # The fp32 convolution the reference's numerics tests run (32-cube).
        dict(kind="conv", name="conv_fp32", n=1, d=32, h=32, w=32, cin=32, cout=32, dtype="fp32"),
        # The up-convolution of a decoder stage (128 -> 64 channels, 32-cube to 64-cube).
        dict(kind="upconv", name="upconv_cube", n=1, d=32, h=32, w=32, cin=128, cout=64, dtype="bf16"),
        # GroupNorm on a mid-level batch of two.
        dict(kind="norm", name="norm_cube", n=2, d=64, h=64, w=64, c=64, dtype="bf16"),
        # GroupNorm at the bottom of the network: the smallest call, all latency.
        dict(kind="norm", name="norm_deep", n=1, d=4, h=8, w=8, c=512, dtype="bf16"),
    ]


def _extent(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choices(("step", "evaluate", "upconv", "conv", "norm"), (9, 3, 2, 5, 3))[0]
    if kind in ("step", "evaluate"):
        base = rng.choice((32, 64))
        # volumes up to the 128-cube, extents even or odd, depth shards thinner than their planes among them
        n, d, h, w = rng.choice((1, 1, 1, 2)), _extent(rng, 16, 128), _extent(rng, 24, 128), _extent(rng, 24, 128)
        # the bottleneck keeps at least four planes, as the network's configuration rule asks for (8 on cubes)
        layers = min(4, max(i for i in (1, 2, 3, 4) if min(d, h, w) >> i >= 4))
        case = dict(kind=kind, n=n, d=d, h=h, w=w, cin=rng.choice((1, 3, 3)), classes=rng.choice((6, 11)), base=base, layers=layers)
        if kind == "step":
            case["halo"] = n == 1 and rng.random() < 0.35
            case["graph"] = rng.random() < 0.35
            case["plain"] = not case["halo"] and not case["graph"] and rng.random() < 0.35
        if n * d * h * w > 128 ** 3:
            case["n"] = 1
        return case
    if kind == "conv":
        dtype = rng.choices(("bf16", "fp16", "fp32"), (6, 2, 2))[0]
        cin = rng.choice((32, 64, 128, 256, 512))
        cout = max(32, min(512, rng.choice((cin // 2, cin, cin, cin * 2))))
        side = {32: 128, 64: 128, 128: 64, 256: 32, 512: 16}[max(cin, cout)]
        if dtype == "fp32":
            side = min(side, 64)
        return dict(kind="conv", n=rng.choice((1, 1, 2)), d=_extent(rng, 4, side), h=_extent(rng, 8, side), w=_extent(rng, 8, side),
                    cin=cin, cout=cout, dtype=dtype)
    if kind == "upconv":
        cin = rng.choice((64, 128, 256, 512))
        side = {64: 64, 128: 32, 256: 16, 512: 8}[cin]
        return dict(kind="upconv", n=rng.choice((1, 1, 2)), d=_extent(rng, 4, side), h=_extent(rng, 4, side), w=_extent(rng, 4, side),
                    cin=cin, cout=cin // 2, dtype=rng.choice(("bf16", "bf16", "fp16")))
    c = rng.choice((32, 64, 128, 256, 512))
    side = {32: 128, 64: 128, 128: 64, 256: 32, 512: 16}[c]
    return dict(kind="norm", n=rng.choice((1, 1, 2)), d=_extent(rng, 4, side), h=_extent(rng, 8, side), w=_extent(rng, 8, side), c=c,
                dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")))


# ---- inputs ----------------------------------------------------------------------------------------------------------
def _fractal_batch(case, g):
    """What the loader hands over on the device: a float32 volume (N, C, D, H, W) and an int16 mask.  Every sample holds the
    voxelised points of three iterated function systems (four affine maps each, contraction 0.3 .. 0.7) of random
    categories; one channel is their occupancy, three are a random colour per category."""
    n, c, d, h, w, classes = (case[k] for k in ("n", "cin", "d", "h", "w", "classes"))
    dev = g.device
    extent = torch.tensor([d, h, w], device=dev, dtype=torch.float32)
    mask = torch.zeros(n, d * h * w, dtype=torch.int16, device=dev)
    chains, keep = 8192, 25
    for i in range(n):
        for _ in range(3):
            r = torch.randn(2, 4, 3, generator=g, device=dev)
            e0 = torch.nn.functional.normalize(r[0], dim=1)
            e1 = torch.nn.functional.normalize(r[1] - (r[1] * e0).sum(1, keepdim=True) * e0, dim=1)
            rotation = torch.stack((e0, e1, torch.linalg.cross(e0, e1)), dim=1)
            maps = rotation * (0.3 + 0.4 * torch.rand(4, 1, 1, generator=g, device=dev))
            shift = torch.rand(4, 3, generator=g, device=dev) - 0.5
            label = torch.randint(1, classes, (1,), generator=g, device=dev).to(torch.int16)
            p = torch.zeros(chains, 3, device=dev)
            points = []
            for t in range(10 + keep):
                k = torch.randint(0, 4, (chains,), generator=g, device=dev)
                p = (maps[k] * p[:, None, :]).sum(-1) + shift[k]
                if t >= 10:
                    points.append(p)
            p = torch.cat(points)
            lo, hi = p.amin(0), p.amax(0)
            at = ((p - lo) / (hi - lo).clamp_min(1e-6) * (extent - 1)).round().long()
            mask[i, (at[:, 0] * h + at[:, 1]) * w + at[:, 2]] = label
    mask = mask.view(n, d, h, w)
    if c == 1:
        volume = (mask > 0).to(torch.float32)[:, None]
    else:
        colours = torch.rand(classes, c, generator=g, device=dev)
        colours[0] = 0
        volume = colours[mask.long()].permute(0, 4, 1, 2, 3)
    return volume.contiguous(), mask


def _unet(case, seed):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = sa.UNet(case["cin"], case["classes"], layers=case["layers"], base_width=case["base"])
    model = model.to(memory_format=CL)
    if case.get("halo"):
        model.set_shard_halo(True)
    if case.get("plain"):
        return model, torch.optim.Adam(model.parameters(), lr=1e-4, fused=True)
    model.defer_weight_gradients(early=True)
    opt = sa.FusedClipAdam(model.parameters(), lr=1e-4, max_norm=1.0, shadow_dtype=torch.bfloat16)
    return model, opt


def _bucket(params):
    """The gradients in one flat buffer, each in its own memory order: what a data-parallel run hands its all-reduce."""
    return torch.cat([(p.grad.permute(0, 2, 3, 4, 1) if p.dim() == 5 else p.grad).reshape(-1) for p in params])


def _train_step(model, opt, params, volume, mask, halo):
    opt.zero_grad(set_to_none=True)
    x, labels = sa.ingest(volume, mask, dtype=torch.bfloat16, out_halo=1 if halo else 0)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = model(x)
    loss = sa.ce_dice_loss(logits, labels)
    loss.backward()
    bucket = _bucket(params)
    opt.step()
    return loss.detach(), logits.detach(), bucket


def _plain_train_step(model, opt, params, volume, mask):
    opt.zero_grad(set_to_none=True)
    x, labels = volume.to(memory_format=CL), mask.to(torch.long)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = model(x)
    loss = sa.ce_dice_loss(logits, labels)
    loss.backward()
    bucket = _bucket(params)
    torch.nn.utils.clip_grad_norm_(params, max_norm=1.0)
    opt.step()
    return loss.detach(), logits.detach(), bucket


def _normal(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=g.device) * scale).to(dtype).contiguous(memory_format=CL)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    n, d, h, w = (case[k] for k in ("n", "d", "h", "w"))
    if kind == "step":
        volume, mask = _fractal_batch(case, g)
        model, opt = _unet(case, seed)
        params = list(model.parameters())
        state = dict(case=case, volume=volume, mask=mask, model=model, opt=opt, params=params)
        if case["graph"]:
            # the program's static input buffers; a batch is copied into them before each replay
            state["in_volume"], state["in_mask"] = volume.clone(), mask.clone()
            args = (model, opt, params, state["in_volume"], state["in_mask"], case["halo"])
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for _ in range(3):
                    _train_step(*args)
            torch.cuda.current_stream().wait_stream(side)
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                state["results"] = _train_step(*args)
        return state
    if kind == "evaluate":
        # between two epochs of a training program: the optimizer has stepped, its bf16 copies of the weights exist
        volume, mask = _fractal_batch(case, g)
        model, opt = _unet(case, seed)
        _train_step(model, opt, list(model.parameters()), volume, mask, False)
        opt.zero_grad(set_to_none=True)
        return dict(case=case, volume=volume, model=model, opt=opt)
    if kind in ("conv", "upconv"):
        dt, cin, cout = DTYPES[case["dtype"]], case["cin"], case["cout"]
        k, up = (3, 1) if kind == "conv" else (2, 2)
        bound = (3.0 / (k ** 3 * cin)) ** 0.5  # Kaiming-uniform over the fan-in
        weight = (torch.rand((cout, cin, k, k, k) if kind == "conv" else (cin, cout, k, k, k), generator=g, device=g.device) * 2 - 1) * bound
        state = dict(case=case, x=_normal(g, (n, cin, d, h, w), dt), gy=_normal(g, (n, cout, d * up, h * up, w * up), dt),
                     w=weight.to(dt).contiguous(memory_format=CL))
        if kind == "upconv":
            state["b"] = torch.randn(cout, generator=g, device=g.device).mul_(bound).to(dt)
        return state
    c, dt = case["c"], DTYPES[case["dtype"]]
    norm = sa.FastGroupNorm(GROUPS, c, activation="relu", device="cuda")
    with torch.no_grad():
        norm.weight.add_(0.1 * torch.randn(c, generator=g, device=g.device))
        norm.bias.add_(0.1 * torch.randn(c, generator=g, device=g.device))
    x = (torch.randn((n, c, d, h, w), generator=g, device=g.device) * 3 + 0.5).to(dt).contiguous(memory_format=CL).requires_grad_()
    return dict(case=case, norm=norm, x=x, gy=_normal(g, (n, c, d, h, w), dt))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        if case["graph"]:
            state["in_volume"].copy_(state["volume"])
            state["in_mask"].copy_(state["mask"])
            state["graph"].replay()
            return state["results"]
        args = (state["model"], state["opt"], state["params"], state["volume"], state["mask"])
        return _plain_train_step(*args) if case["plain"] else _train_step(*args, case["halo"])
    if kind == "evaluate":
        with torch.no_grad():
            x, _ = sa.ingest(state["volume"], dtype=torch.bfloat16)
            with torch.autocast("cuda", dtype=torch.bfloat16):
                return state["model"](x)
    if kind == "conv":
        x, w, gy = state["x"], state["w"], state["gy"]
        return (sa.conv3d_forward(x, w, None, 1, 1), sa.conv3d_backward_data(gy, w, x.shape, 1, 1),
                sa.conv3d_backward_weight(x, w.shape, gy, 1, 1))
    if kind == "upconv":
        x, w, gy = state["x"], state["w"], state["gy"]
        return (sa.conv_transpose3d_forward(x, w, state["b"], 2), sa.conv_transpose3d_backward_data(gy, w, x.shape, 2),
                sa.conv_transpose3d_backward_weight(x, w.shape, gy, 2))
    norm, x = state["norm"], state["x"]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=x.dtype is not torch.float32):
        y = norm(x)
    return (y.detach(), *torch.autograd.grad(y, (x, norm.weight, norm.bias), state["gy"]))


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
def _conv_work(vox_in, vox_out, cin, cout, taps, es, passes):
    """(bytes, flops) of ``passes`` directions of one convolution: every direction reads its two operands and writes its
    result once; ``passes`` = 1 forward, 2 without the data gradient (the network's first convolution), 3 all."""
    x, y, wt = vox_in * cin * es, vox_out * cout * es, taps * cin * cout * es
    return (x + y + wt) * passes, 2.0 * vox_out * cin * cout * taps * passes


def _network_work(case, train):
    n, cin, classes, base, layers = (case[k] for k in ("n", "cin", "classes", "base", "layers"))
    dims = [(case["d"], case["h"], case["w"])]
    for _ in range(layers):
        dims.append(tuple(v // 2 for v in dims[-1]))
    vox = [n * a * b * c for a, b, c in dims]
    full, es = (3 if train else 1), 2
    total_b, total_f, params = vox[0] * (4 * cin + es * cin + 10), 0.0, 0

    def add(bf, weights=0):
        nonlocal total_b, total_f, params
        total_b, total_f, params = total_b + bf[0], total_f + bf[1], params + weights

    def double(v, ci, co, first=False):
        for a in (ci, co):
            add(_conv_work(v, v, a, co, 27, es, 2 if (train and first and a == ci) else full), 27 * a * co)
            # normalisation: x in, y out; backward x and dy in, dx out
            add((v * co * es * (5 if train else 2), 8.0 * v * co * full), 2 * co)

    for i in range(layers + 1):
        c = base << i
        if i:
            # pooling: x in, y out; backward dy in, dx out
            add(((vox[i - 1] + vox[i]) * (c // 2) * es * (2 if train else 1), 8.0 * vox[i] * (c // 2)))
        double(vox[i], cin if i == 0 else c // 2, c, first=i == 0)
    for i in range(layers, 0, -1):
        c = base << i
        add(_conv_work(vox[i], vox[i] * 8, c, c // 2, 1, es, full), 8 * c * (c // 2))
        double(vox[i - 1], c, c // 2)
    add(_conv_work(vox[0], vox[0], base, classes, 1, es, full), base * classes)
    if train:
        total_b += vox[0] * (4 * classes + 16)  # the loss reads logits and labels, its gradient both again and writes one
        total_b += params * 34  # clip + Adam: gradient twice, weight and moments read and written, 16-bit copy
    return {"bytes": float(total_b), "flops": float(total_f)}


def work(case):
    kind = case["kind"]
    if kind in ("step", "evaluate"):
        return _network_work(case, kind == "step")
    n, d, h, w = (case[k] for k in ("n", "d", "h", "w"))
    v = n * d * h * w
    if kind == "conv":
        es = 4 if case["dtype"] == "fp32" else 2
        b, f = _conv_work(v, v, case["cin"], case["cout"], 27, es, 3)
        return {"bytes": float(b), "flops": f}
    if kind == "upconv":
        # a small voxel and tap meet in one of the eight output voxels
        b, f = _conv_work(v, 8 * v, case["cin"], case["cout"], 1, 2, 3)
        return {"bytes": float(b), "flops": f}
    es = 4 if case["dtype"] == "fp32" else 2
    return {"bytes": float(v * case["c"] * es * 5), "flops": 24.0 * v * case["c"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("step", "evaluate"):
        # against the same network from stock modules under the same autocast (every rounding in another place): logits
        # 5e-3 to 6e-3, flat gradient 2e-3, loss 2e-5
        return {"rel": 2e-2}
    # operators against a 64-bit run of the same operands: bf16 1.7e-3, fp16 2.1e-4 (the rounding of the results),
    # fp32 5e-7 for the convolutions and 1.5e-7 for the normalisation
    rel = {"bf16": 7e-3, "fp16": 1e-3, "fp32": 2e-6}[case["dtype"]]
    if kind == "norm":
        # an element whose pre-activation is zero to the last bit may pass the ReLU in one implementation and not in another
        return {"rel": rel, "max": 0.99}
    return {"rel": rel}
