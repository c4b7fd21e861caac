"""The work a user of this framework has it do, as cases that can be timed and compared.

A case is one call of a user's program on a transcoder that the program keeps: a forward (``model(inputs)`` under
``no_grad``), dense activations for analysis (``get_feature_activations``), one optimisation step
(``training_step`` with ``CLTAdam``), or a forward and backward through autograd.  The listed cases carry the sizes
of ``synth.WORKLOADS`` (C0 - C3 of the benchmark), the smoke test's model and two generic ones; ``draw`` spreads
over the ranges they stand for.

Keys of a case
    op           "forward", "features", "train" or "autograd"
    L, d, F, T   layers, d_model, features per layer, tokens of the batch
    dtype        element type of the model
    fn           "batchtopk" (k survivors per token on average, over a layer or over all layers), "topk"
                 (exactly k per token) or "jumprelu" (about 0.6 % of the features fire per token)
    k, scope     survivors per token and what they are counted over ("per_layer" or "global"; top-k family only)
    tying        decoders: "none" (one per source and target), "per_source" or "per_target"
"""

import torch

import crosslayer_coding_amd as cca
from crosslayer_coding_amd import synth

JUMPRELU_DENSITY = 0.006        # what synth calibrates the thresholds to


def _case(name, op, L, d, F, T, dtype="bfloat16", fn="batchtopk", k=200, scope="per_layer", tying="none"):
    case = {"op": op, "L": L, "d": d, "F": F, "T": T, "dtype": dtype, "fn": fn, "k": 0 if fn == "jumprelu" else k,
            "scope": scope, "tying": tying}
    return dict(case, name=name) if name else case


def listed():
    return [
        # a toy model in a unit test or a notebook: launches and host work are all of it
        _case("forward_tiny", "forward", 3, 768, 1024, 32, "float32", k=16),
        # one short prompt through a full-size transcoder: interactive attribution, token by token reading
        _case("forward_prompt", "forward", 12, 768, 24576, 77),
        # a small transcoder kept in float32, the configuration's default type
        _case("forward_c0", "forward", 12, 768, 6144, 1024, "float32"),
        # the headline: batches of activations through a GPT-2-small x32 transcoder
        _case("forward_c1", "forward", 12, 768, 24576, 4096),
        # the scope a configuration has unless it says otherwise, on a batch that is no whole number of tiles
        _case("forward_global", "forward", 12, 768, 24576, 3000, scope="global"),
        # thresholds in place of top-k: what a trained transcoder is converted to for use; the largest decoder set
        _case("forward_jumprelu", "forward", 24, 1024, 32768, 4096, fn="jumprelu"),
        # one decoder per target layer: the matrix-core formulation of the decode
        _case("forward_per_target", "forward", 16, 2048, 16384, 8192, tying="per_target"),
        # dense activations of every layer, for dashboards and circuit analysis
        _case("features", "features", 12, 768, 24576, 1000),
        # training at the headline size: forward, loss, gradients and Adam
        _case("train_c1", "train", 12, 768, 24576, 4096),
        # training a small transcoder in float32
        _case("train_c0", "train", 12, 768, 6144, 1024, "float32"),
        # training in the default scope on a ragged batch, a wider model with fewer layers
        _case("train_global", "train", 6, 1024, 16384, 1500, scope="global"),
        # a caller's own loss on the reconstructions: forward and backward through autograd, thresholds learned too
        _case("autograd_jumprelu", "autograd", 6, 512, 16384, 2048, fn="jumprelu"),
    ]


def _log_between(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["forward", "forward", "forward", "features", "train", "train", "autograd"])
    d = rng.choice([256, 512, 640, 768, 1024, 2048])
    # autograd hands every parameter's gradient back separately: models of few layers
    L = rng.randint(2, 6) if op == "autograd" else rng.randint(2, 16)
    F = 8 * _log_between(rng, 1024 // 8, 32768 // 8)
    T = _log_between(rng, 32, 8192)
    dtype = rng.choice(["bfloat16", "bfloat16", "bfloat16", "float32"] + (["float16"] if op in ("forward", "features") else []))
    fn = rng.choice(["batchtopk", "batchtopk", "batchtopk", "jumprelu", "topk"])
    scope = rng.choice(["per_layer", "global"])
    k = _log_between(rng, 16, max(17, min(256, F // 50)))
    tying = rng.choice(["none", "none", "none", "per_source", "per_target"])
    # no drawn case is larger than the largest listed one: halve the batch, then the features, until it is not
    def size(T_, F_):
        return L * T_ * F_ * (d + 512), L * (L + 1) // 2 * F_ * d * (3 if op == "train" else 1)
    while (size(T, F)[0] > 2.5e12 or size(T, F)[1] > 1.5e9) and F > 1024:
        if size(T, F)[1] > 1.5e9 or T < 64:
            F = 8 * (F // 16)
        else:
            T = (T + 1) // 2
    return _case(None, op, L, d, F, T, dtype, fn, min(k, F // 8), scope, tying)


def _workload(case):
    return synth.Workload("case", 0, case["L"], case["d"], case["F"], case["T"], case["dtype"], case["fn"],
                          case["k"] or None, case["scope"], case["tying"])


class _State:
    pass


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    wl = _workload(case)
    st = _State()
    st.case = case
    st.model, st.inputs, _ = synth.build_model(wl, dev, seed)
    st.targets = st.optimizer = st.params = None
    if case["op"] in ("train", "autograd"):
        y = synth.make_targets(wl, dev, seed)
        st.targets = {l: y[l] for l in range(wl.num_layers)}
    if case["op"] == "train":
        st.optimizer = cca.CLTAdam(st.model, lr=1e-4)
    if case["op"] == "autograd":
        st.params = [p for _, p in st.model.named_parameters() if p.requires_grad]
    return st


def run(st):
    op, model = st.case["op"], st.model
    if op == "forward":
        with torch.no_grad():
            return model(st.inputs)
    if op == "features":
        with torch.no_grad():
            return model.get_feature_activations(st.inputs)
    if op == "train":
        loss = model.training_step(st.inputs, st.targets, st.optimizer)
        # the step's results: the updated weights (encoders stacked, decoders feature-major) and the moments of the
        # encoders and of every bias, which hold their gradients
        w_enc, b_enc = model.encoder_module.stacked()
        state = st.optimizer.state
        return {"loss": loss, "enc_w": w_enc, "enc_b": b_enc, "dec_w": model.decoder_module.packed(),
                "m_enc_w": state["enc_w"][0], "m_enc_b": state["enc_b"][0], "m_dec_b": state["dec_b"][0]}
    for p in st.params:
        p.grad = None
    recs = model(st.inputs)
    loss = sum(torch.nn.functional.mse_loss(recs[l].float(), st.targets[l].float()) for l in recs)
    loss.backward()
    return [loss.detach()] + [p.grad for p in st.params if p.grad is not None]


def _survivors(case):
    """Survivors of all layers together."""
    if case["fn"] == "jumprelu":
        return JUMPRELU_DENSITY * case["L"] * case["T"] * case["F"]
    return case["k"] * case["T"] * (case["L"] if case["scope"] == "per_layer" else 1)


def work(case):
    """Bytes and operations one pass cannot do without, weights and tensors counted once each."""
    L, d, F, T, op = case["L"], case["d"], case["F"], case["T"], case["op"]
    e = 4 if case["dtype"] == "float32" else 2
    n = _survivors(case)
    n_dec = L * (L + 1) // 2 if case["tying"] == "none" else L
    enc_flops = 2.0 * T * d * F * L
    io = L * T * d * e
    enc_bytes = L * F * d * e + io
    if op == "features":
        return {"bytes": enc_bytes + L * T * F * (4 if case["fn"] == "jumprelu" else e), "flops": enc_flops}
    # a survivor of source s adds one decoder row to every target >= s; per target tying sums the sources first
    rows = n * (L + 1) / 2.0
    dec_flops = 2.0 * rows * d if case["tying"] == "none" else 2.0 * n * d
    # decoder rows that at least one survivor needs
    used = F * (1.0 - (1.0 - min(1.0, n / (L * T * F))) ** T)
    dec_bytes = n_dec * used * d * e
    if op == "forward":
        return {"bytes": enc_bytes + dec_bytes + io, "flops": enc_flops + dec_flops}
    # backward: gradient of the kept activations and of the decoders, each as much as the decode; of the encoders
    flops = enc_flops + 3.0 * dec_flops + 2.0 * n * d
    moved = enc_bytes + dec_bytes + 3 * io
    params = (n_dec + L) * F * d
    if op == "train":
        moved += params * (2 * e + 16.0) - n_dec * used * d * e      # weights and both moments read and written
    else:
        moved += params * e                                          # every gradient written
        if case["fn"] == "jumprelu":
            # the threshold gradient needs d loss / d activation on both sides of the threshold
            flops += 2.0 * T * F * d * n_dec
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # Measured by running every listed and several drawn cases against themselves with the encoder's sum over d_model
    # in another order, and stated about four times as wide.  Few pre-activations round differently then, but those at
    # a selection threshold change places: rel 1.2e-3 .. 2.7e-3 of the reconstructions and activations (float32 too),
    # 1.5e-3 .. 4.9e-3 of a training step's results; a single value that changes places is off by its whole size.
    if case["op"] == "train":
        return {"rel": 2e-2 if case["scope"] == "global" else 1e-2, "max": 0.99}
    if case["op"] == "features":
        return {"rel": 1.2e-2, "max": 0.99}
    if case["dtype"] == "float32":
        return {"rel": 5e-3, "max": 0.5}
    return {"rel": 1e-2, "max": 0.8}
