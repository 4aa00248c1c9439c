"""The work that users of this framework have it do, as cases that can be timed and checked.

One pass of a case is one call (for the real convolution with fresh filters, two) of a
public entry point of thunderfft_amd on device buffers that the caller owns.  Complex
values are real-imaginary pairs in the last axis, in float32 or float16.

op        what a pass does
c2c       ThunderFFT_global_async, or ThunderFFT_global (which waits) where "wait" is set;
          "offset" elements between the 16-byte boundary and the buffers' start
conv1d    ThunderFFT_conv1d_async, one filter per signal or one for all
real      ThunderFFT_conv1d_real_async of [batch][channels][n] samples; with "filters" the
          channel spectra are made anew in the pass (ThunderFFT_conv1d_real_filter_async)
valid     ThunderFFT_conv1d_valid_async of `batch` signals of `n` values with `taps` taps
conv2d    ThunderFFT_conv2d_async of `batch` n x n images with one filter
"""
import math

import torch

import thunderfft_amd as thff

LENGTHS = thff.SUPPORTED_N
_DTYPE = {"float": torch.float32, "half": torch.float16}


def listed():
    return [
        # The quick start's call: 16 signals of 64, waited for.  Latency only.
        dict(name="c2c_f32_n64_b16", op="c2c", T="float", n=64, batch=16, forward=True, wait=True, offset=0),
        # The headline batch, one GiB of traffic.
        dict(name="c2c_f32_n1024_b65536", op="c2c", T="float", n=1024, batch=65536, forward=True, wait=False, offset=0),
        # An ordinary batch of the longest transform, back from the spectrum, not a multiple of anything.
        dict(name="c2c_f16_n4096_b1001", op="c2c", T="half", n=4096, batch=1001, forward=False, wait=False, offset=0),
        # Fused convolution with a filter for each signal, the benchmark's shape.
        dict(name="conv1d_f32_n2048_b16384", op="conv1d", T="float", n=2048, batch=16384, per_signal=True),
        # Fused convolution of an ordinary ragged batch with one filter for all.
        dict(name="conv1d_f16_n1024_b4099", op="conv1d", T="half", n=1024, batch=4099, per_signal=False),
        # Long-convolution layer (half, 64 channels) whose filters changed since the last step.
        dict(name="real_f16_n4096_256x64", op="real", T="half", n=4096, batch=256, channels=64, filters=True),
        # The same layer in float at an ordinary size, odd batch, filters kept.
        dict(name="real_f32_n512_33x96", op="real", T="float", n=512, batch=33, channels=96, filters=False),
        # One long recording against a short filter, the benchmark's shape.
        dict(name="valid_f32_2e26_t9", op="valid", T="float", n=1 << 26, batch=1, taps=9),
        # A batch of recordings of odd length against a longer filter.
        dict(name="valid_f16_100003x64_t41", op="valid", T="half", n=100003, batch=64, taps=41),
        # Many small images, the benchmark's shape.
        dict(name="conv2d_f32_64_b8192", op="conv2d", T="float", n=64, batch=8192),
        # The reference sample's single large image, in half.
        dict(name="conv2d_f16_1024_b1", op="conv2d", T="half", n=1024, batch=1),
        # A batch of large images, the most that a pass here does.
        dict(name="conv2d_f32_1024_b32", op="conv2d", T="float", n=1024, batch=32),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["c2c", "c2c", "c2c", "conv1d", "conv1d", "real", "real", "valid", "valid", "conv2d", "conv2d"])
    T = rng.choice(["float", "half"])
    n = rng.choice(LENGTHS)
    if op == "c2c":
        batch = max(1, _log_uniform(rng, 1 << 10, 1 << 26) // n)
        # One call in eight is on a slice that starts inside a 16-byte vector.
        return dict(op=op, T=T, n=n, batch=batch, forward=rng.random() < 0.5, wait=rng.random() < 0.25,
                    offset=1 if rng.random() < 0.125 else 0)
    if op == "conv1d":
        batch = max(1, _log_uniform(rng, 1 << 12, 1 << 25) // n)
        return dict(op=op, T=T, n=n, batch=batch, per_signal=rng.random() < 0.5)
    if op == "real":
        channels = _log_uniform(rng, 1, 768)
        batch = max(1, _log_uniform(rng, 1 << 14, 1 << 26) // (n * channels))
        return dict(op=op, T=T, n=n, batch=batch, channels=channels, filters=rng.random() < 0.3)
    if op == "valid":
        taps = rng.randint(1, 64)
        # Long filters over shorter recordings, so that none costs more than the listed cases.
        values = _log_uniform(rng, 1 << 12, max(1 << 13, (1 << 26) * (65 - taps) // 64))
        batch = min(_log_uniform(rng, 1, 256), values // 1024)
        return dict(op=op, T=T, n=values // batch, batch=batch, taps=taps)
    n = rng.choice([64, 128, 1024])
    return dict(op=op, T=T, n=n, batch=max(1, _log_uniform(rng, 1 << 16, 1 << 25) // (n * n)))


def _outputs(case):
    """(values of the output, numbers per value)"""
    if case["op"] == "real":
        return case["batch"] * case["channels"] * case["n"], 1
    if case["op"] == "valid":
        return case["batch"] * (case["n"] - case["taps"] + 1), 2
    if case["op"] == "conv2d":
        return case["batch"] * case["n"] ** 2, 2
    return case["batch"] * case["n"], 2


def _shape(case):
    if case["op"] == "real":
        return (case["batch"], case["channels"], case["n"])
    if case["op"] == "valid":
        return (case["batch"], case["n"] - case["taps"] + 1, 2)
    if case["op"] == "conv2d":
        return (case["batch"], case["n"], case["n"], 2)
    return (case["batch"], case["n"], 2)


def _inputs(case, seed):
    """The signals x and the filter h of a case, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    op, n, batch, dtype = case["op"], case["n"], case["batch"], _DTYPE[case["T"]]

    def normal(*shape, dtype=dtype, scale=1.0):
        v = torch.randn(*shape, device="cuda", generator=gen)
        return v.mul_(scale).to(dtype)

    if op == "c2c":
        return normal(batch, n, 2), None
    if op == "conv1d":
        return normal(batch, n, 2), normal(batch if case["per_signal"] else 1, n, 2, scale=1 / math.sqrt(n))
    if op == "real":
        # Decaying filters over the whole length, as a long-convolution layer has.
        decay = torch.exp(-4.0 * torch.arange(n, device="cuda") / n)
        h = normal(case["channels"], n, dtype=torch.float32, scale=1 / math.sqrt(n))
        return normal(batch, case["channels"], n), h.mul_(decay)
    if op == "valid":
        return normal(batch, n, 2), normal(case["taps"], 2, dtype=torch.float32, scale=1 / math.sqrt(case["taps"]))
    # A real 7 x 7 kernel in the corner of an otherwise empty filter.
    h = torch.zeros(n, n, 2, device="cuda")
    h[:7, :7, 0] = normal(7, 7, dtype=torch.float32, scale=1 / 7)
    return normal(batch, n, n, 2), h.to(dtype)


def prepare(case, seed):
    thff.ThunderFFTInitialize(case["T"], 64 if case["op"] == "valid" else case["n"])
    x, h = _inputs(case, seed)
    y = torch.empty(_shape(case), dtype=x.dtype, device="cuda")
    state = dict(case=case, x=x, h=h, y=y)
    offset = case.get("offset", 0)
    if offset:  # both buffers become slices that start `offset` values into a larger one
        for key in ("x", "y"):
            t = state[key]
            whole = torch.empty(t.numel() + 2 * offset, dtype=t.dtype, device="cuda")
            part = whole[2 * offset:].view(t.shape)
            part.copy_(t)
            state[key] = part
    if case["op"] == "real":
        state["spectrum"] = torch.empty(case["channels"], case["n"], 2, device="cuda")
        if not case["filters"]:
            thff.ThunderFFT_conv1d_real_filter(case["T"], case["n"], h, state["spectrum"], case["channels"],
                                               1.0 / case["n"], torch.cuda.current_stream())
    return state


def run(state):
    case, x, h, y = state["case"], state["x"], state["h"], state["y"]
    op, T, n, batch = case["op"], case["T"], case["n"], case["batch"]
    stream = torch.cuda.current_stream()
    if op == "c2c":
        call = thff.ThunderFFT_global if case["wait"] else thff.ThunderFFT_global_async
        call(T, n, case["forward"], x, y, batch, stream)
    elif op == "conv1d":
        thff.ThunderFFT_conv1d_async(T, n, x, h, y, batch, case["per_signal"], stream)
    elif op == "real":
        spectrum = state["spectrum"]
        if case["filters"]:
            thff.ThunderFFT_conv1d_real_filter_async(T, n, h, spectrum, case["channels"], 1.0 / n, stream)
        thff.ThunderFFT_conv1d_real_async(T, n, x, spectrum, y, batch, case["channels"], stream)
    elif op == "valid":
        thff.ThunderFFT_conv1d_valid_async(T, x, n, h, case["taps"], y, batch, stream)
    else:
        thff.ThunderFFT_conv2d_async(T, n, n, x, h, y, batch, stream)
    return y


def work(case):
    """Signals and filters read once, results written once; 5 N log2 N for a complex
    transform of N, half of that for a real one, 6 for a complex product."""
    op, n, batch = case["op"], case["n"], case["batch"]
    size = 4 if case["T"] == "float" else 2
    values, per = _outputs(case)
    written = values * per * size
    if op == "c2c":
        return dict(bytes=2 * written, flops=5 * values * math.log2(n))
    if op == "conv1d":
        filters = batch if case["per_signal"] else 1
        return dict(bytes=2 * written + filters * n * 2 * size,
                    flops=5 * n * math.log2(n) * (2 * batch + filters) + 6 * values)
    if op == "real":
        taps = case["channels"] * n
        # Fresh filters are read as taps, kept ones as spectra (half of each is redundant).
        return dict(bytes=2 * written + 4 * taps,
                    flops=5 * math.log2(n) * values + 3 * values
                    + (2.5 * math.log2(n) * taps if case["filters"] else 0))
    if op == "valid":
        read = batch * n * per * size + 8 * case["taps"]
        # The direct sum, or two transforms of 256 for 257 - taps outputs, whichever is less.
        each = min(8 * case["taps"], (2 * 5 * 256 * 8 + 6 * 256) / (257 - case["taps"]))
        return dict(bytes=read + written, flops=each * values)
    return dict(bytes=2 * written + n * n * 2 * size,
                flops=2 * 5 * math.log2(n * n) * values + 5 * n * n * math.log2(n * n) + 6 * values)


def tolerance(case):
    """About four times the error against 64 bits that was measured: 1e-7 to 3e-7 in float
    (the direct sums and the transforms of 64 least, the convolutions most); in half 2e-4
    to 4e-4 for a transform and 3e-4 to 9e-4 for a convolution, whose values are rounded
    to 16 bits between the stages."""
    if case["T"] == "float":
        return dict(rel=1.2e-6)
    return dict(rel=1.6e-3 if case["op"] == "c2c" else 3.5e-3)


def exact(case, seed):
    x, h = _inputs(case, seed)
    op, n, batch = case["op"], case["n"], case["batch"]
    out = torch.empty(_shape(case), dtype=torch.float64, device="cuda")

    def complex_(v):
        return torch.view_as_complex(v.to(torch.float64))

    # In pieces, so that the work in 64 bits needs little memory.
    if op == "valid":
        taps = complex_(h)
        step = 1 << 22
        count = n - case["taps"] + 1
        for b in range(batch):
            for i in range(0, count, step):
                m = min(step, count - i)
                part = complex_(x[b, i:i + m + case["taps"] - 1])
                got = torch.zeros(m, dtype=torch.complex128, device="cuda")
                for k in range(case["taps"]):
                    got += part[k:k + m] * taps[k]
                out[b, i:i + m] = torch.view_as_real(got)
        return out
    step = max(1, (1 << 24) // (n * n if op == "conv2d" else n * case.get("channels", 1)))
    if op == "conv2d":
        H = torch.fft.fft2(complex_(h))
    elif op == "real":
        H = torch.fft.rfft(h.to(torch.float64))
    elif op == "conv1d" and not case["per_signal"]:
        H = torch.fft.fft(complex_(h))
    for b in range(0, batch, step):
        part = x[b:b + step]
        if op == "c2c":
            v = complex_(part)
            got = torch.fft.fft(v) if case["forward"] else torch.fft.ifft(v, norm="forward")
        elif op == "conv1d":
            spectrum = torch.fft.fft(complex_(h[b:b + step])) if case["per_signal"] else H
            got = torch.fft.ifft(torch.fft.fft(complex_(part)) * spectrum)
        elif op == "real":
            out[b:b + step] = torch.fft.irfft(torch.fft.rfft(part.to(torch.float64)) * H, n)
            continue
        else:
            got = torch.fft.ifft2(torch.fft.fft2(complex_(part)) * H)
        out[b:b + step] = torch.view_as_real(got)
    return out
