"""What the speed of this package is measured on: passes a user's program makes through the public entry points.

A case is one pass of one ``path``:

* ``dynamics``  -- the operators one by one, as the reference's neuron classes call them: leaky integrator, leaky
  integrator with reset, spike; forward only or forward and backward down to the gradients of the input and of both
  decays;
* ``neuron``    -- a CUBA, ALIF or RF neuron module, forward only or as a training step (``learn``: its decays are
  trained, so they receive gradients too);
* ``block``     -- temporal filter, CUBA neuron and the learnable axonal delay behind it, with the gradients of the
  input and of the delays;
* ``conv``      -- convolution synapse and CUBA neuron, the layer convolutional spiking networks are stacked from, with
  the gradients of the input spikes and of the weights;
* ``decoder``   -- pooling and transposed-convolution synapses (down and up again), with the same gradients;
* ``dense``     -- dense synapse and CUBA neuron;
* ``recurrent`` -- a recurrent CUBA or ALIF layer.

Inputs are what such layers meet: sparse spikes or weighted sparse events, normally distributed upstream gradients,
synapse weights on the 8-bit grid of the neuron's quantiser (so weighted spikes are exact in float32 in any order of
summation and the spike trains do not depend on it).  All of it is drawn on the GPU from the seed alone.
"""
import math

import torch

import lava_dl_amd.slayer as slayer

DEVICE = 'cuda'


def listed():
    return [
        # one small batch through the dynamics operators, nothing to differentiate: 512 neurons, what a launch and a
        # sequential step cost
        dict(name='dynamics_small_forward', path='dynamics', train=False, batch=4, shape='128', steps=200),
        # the neuron tensor of a convolutional layer through the operators one by one, as a training step
        dict(name='dynamics_conv_train', path='dynamics', train=True, batch=32, shape='16x32x32', steps=300),
        # a dense layer's neurons over samples whose length is not a multiple of four steps, decays trained
        dict(name='cuba_ragged_train', path='neuron', model='cuba', train=True, learn=True, graded=False, batch=16,
             shape='512', steps=1450),
        # adaptive-threshold neurons with fixed decays, the module's default
        dict(name='alif_train', path='neuron', model='alif', train=True, learn=False, graded=False, batch=64,
             shape='512', steps=1000),
        # resonators over long samples, rotation parameters trained: the largest tensors of the list
        dict(name='rf_train', path='neuron', model='rf', train=True, learn=True, graded=False, batch=64, shape='1024',
             steps=2000),
        # synaptic filter, neuron and trained axonal delay: the stack of a dense layer with temporal kernels
        dict(name='block_train', path='block', train=True, taps=64, batch=32, shape='256', steps=1500),
        # the first convolutional layer of a network: few input channels, memory-bound
        dict(name='conv_train', path='conv', train=True, batch=32, inputs=8, outputs=16, height=32, width=32, kernel=3,
             stride=1, padding=1, steps=300),
        # a deeper, wider layer: more arithmetic per byte
        dict(name='conv_wide_train', path='conv', train=True, batch=16, inputs=32, outputs=64, height=16, width=16,
             kernel=3, stride=1, padding=1, steps=300),
        # down by two with pooling and up again with a transposed convolution, as in an auto-encoder
        dict(name='decoder_train', path='decoder', train=True, batch=32, inputs=16, outputs=8, height=32, width=32,
             steps=300),
        # a dense layer at inference
        dict(name='dense_forward', path='dense', train=False, batch=32, inputs=256, outputs=256, steps=1500),
        # a wide recurrent layer
        dict(name='recurrent_wide_train', path='recurrent', model='cuba', train=True, batch=32, neurons=2048, steps=300),
        # a narrow one, the size recurrent layers of small networks have
        dict(name='recurrent_narrow_train', path='recurrent', model='alif', train=True, batch=32, neurons=128, steps=300),
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _steps(rng, lo, hi):
    """Sample lengths: any number of steps, or the round ones that data sets are cut to."""
    grain = rng.choice((1, 2, 4, 50))
    return max(lo, min(hi, _log_uniform(rng, lo, hi) // grain * grain))


def _neurons(rng, batch, steps, most, image):
    """Neurons of one sample (flat or C x H x W) such that the tensor holds 100 thousand to ``most`` samples."""
    per_sample = max(8, _log_uniform(rng, 100000, most) // (batch * steps))
    if not image or per_sample < 4 * 64:
        return str(min(per_sample, 65536))
    side = rng.randint(8, 34)
    channels = max(1, min(64, per_sample // (side * side)))
    return f'{channels}x{side}x{side}'


def draw(rng):
    path = rng.choice(('dynamics', 'neuron', 'neuron', 'neuron', 'block', 'conv', 'conv', 'decoder', 'dense',
                       'recurrent', 'recurrent'))
    train = rng.random() < 0.75
    batch = _log_uniform(rng, 1, 64)
    if path == 'dynamics':
        steps = _steps(rng, 100, 2000)
        return dict(path=path, train=train, batch=batch, steps=steps,
                    shape=_neurons(rng, batch, steps, 150000000, rng.random() < 0.5))
    if path == 'neuron':
        model = rng.choice(('cuba', 'alif', 'rf'))
        steps = _steps(rng, 100, 2000)
        return dict(path=path, model=model, train=train, learn=model != 'alif' and rng.random() < 0.5,
                    graded=rng.random() < 0.2, batch=batch, steps=steps,
                    shape=_neurons(rng, batch, steps, {'cuba': 150000000, 'alif': 60000000, 'rf': 130000000}[model],
                                   rng.random() < 0.4))
    if path == 'block':
        steps = _steps(rng, 200, 1500)
        return dict(path=path, train=train, taps=_log_uniform(rng, 10, 100), batch=batch, steps=steps,
                    shape=_neurons(rng, batch, steps, 40000000, False))
    if path == 'conv':
        batch, steps = _log_uniform(rng, 4, 32), _steps(rng, 50, 350)
        kernel, inputs, side = rng.choice((3, 3, 5)), rng.choice((2, 4, 8, 16, 32)), rng.randint(8, 34)
        outputs = min(64, 2 * inputs if inputs > 2 else rng.choice((8, 16)))
        # pixels times steps: what the two tensors hold, and what the products cost
        most = min(470000000 // (inputs + outputs), 22000000000 // (inputs * outputs * kernel ** 2))
        if batch * side * side * steps > most:
            batch = max(1, most // (side * side * steps))
        return dict(path=path, train=train, batch=batch, inputs=inputs, outputs=outputs, height=side,
                    width=max(8, side - rng.randint(0, 3)), kernel=kernel, stride=rng.choice((1, 1, 2)),
                    padding=kernel // 2, steps=steps)
    if path == 'decoder':
        batch, steps = _log_uniform(rng, 4, 32), _steps(rng, 50, 350)
        return dict(path=path, train=train, batch=batch, inputs=rng.choice((4, 8, 16)), outputs=rng.choice((2, 4, 8)),
                    height=2 * rng.randint(4, 16), width=2 * rng.randint(4, 16), steps=steps)
    if path == 'dense':
        inputs, outputs, steps = _log_uniform(rng, 64, 1024), _log_uniform(rng, 16, 1024), _steps(rng, 100, 1500)
        return dict(path=path, train=train, batch=max(1, min(batch, 16000000000 // (inputs * outputs * steps))),
                    inputs=inputs, outputs=outputs, steps=steps)
    wide = rng.random() < 0.6
    return dict(path=path, model=rng.choice(('cuba', 'alif')), train=train, batch=_log_uniform(rng, 8, 32),
                neurons=4 * _log_uniform(rng, 64, 512) if wide else _log_uniform(rng, 32, 256),
                steps=_steps(rng, 50, 300))


# ------------------------------------------------------------------------------------------------ state
def _dims(case):
    return tuple(int(d) for d in case['shape'].split('x'))


def _events(gen, shape, rate, amplitude):
    """Sparse weighted events: Bernoulli(rate) times N(0, amplitude)."""
    x = torch.randn(shape, generator=gen, device=DEVICE).mul_(amplitude)
    return x.mul_(torch.rand(shape, generator=gen, device=DEVICE) < rate)


def _spikes(gen, shape, rate):
    return (torch.rand(shape, generator=gen, device=DEVICE) < rate).float()


def _weights(gen, synapse, std):
    synapse.weight.data = torch.randn(synapse.weight.shape, generator=gen, device=DEVICE) * std


def _settled(neuron, *input):
    """The module after its first call, which fixes its shape and draws its per-channel parameters."""
    with torch.no_grad():
        neuron(input if len(input) > 1 else input[0])
    return neuron


def prepare(case, seed):
    torch.manual_seed(seed)                       # the neuron modules draw their per-channel parameters from it
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    path, train, steps, batch = case['path'], case['train'], case['steps'], case['batch']
    st = dict(case=case)

    def random(*shape):
        return torch.randn(shape, generator=gen, device=DEVICE)

    def decays(count):
        return torch.randint(0, 4096, (count,), generator=gen, device=DEVICE).float()

    if path == 'dynamics':
        dims = _dims(case)
        st.update(x=_events(gen, (batch,) + dims + (steps,), 0.02 if train else 0.05, 0.5 if train else 1.0),
                  current_decay=decays(dims[0]) if train else torch.full((1,), 1024.0, device=DEVICE),
                  voltage_decay=decays(dims[0]) if train else torch.full((1,), 128.0, device=DEVICE),
                  state=torch.zeros(1, device=DEVICE), threshold=1.0 if train else 1.25)
        wrt = ['x', 'current_decay', 'voltage_decay']
        out_shape = st['x'].shape
    elif path == 'neuron':
        shape = (batch,) + _dims(case) + (steps,)
        common = dict(shared_param=False, requires_grad=case['learn'], graded_spike=case['graded'])
        if case['model'] == 'rf':
            st.update(x=_events(gen, shape, 0.1, 0.3), x_imag=_events(gen, shape, 0.1, 0.3))
            neuron = slayer.neuron.rf.Neuron(threshold=1.0, period=[20, 200], decay=[0.01, 0.9], **common)
        elif case['model'] == 'alif':
            st.update(x=_events(gen, shape, 0.05, 1.0))
            neuron = slayer.neuron.alif.Neuron(threshold=1.0, threshold_step=0.5, current_decay=[0, 1],
                                               voltage_decay=[0, 1], threshold_decay=[0, 1], refractory_decay=[0, 1],
                                               **common)
        else:
            st.update(x=_events(gen, shape, 0.05, 0.5))
            neuron = slayer.neuron.cuba.Neuron(threshold=1.0, current_decay=[0, 1], voltage_decay=[0, 1], **common)
        inputs = [st[k] for k in ('x', 'x_imag') if k in st]
        st['neuron'] = _settled(neuron.to(DEVICE), *inputs)
        wrt = ['x', 'x_imag'][:len(inputs)]
        if case['learn']:
            st.update(neuron.named_parameters(recurse=False))
            wrt += [k for k, _ in neuron.named_parameters(recurse=False)]
        out_shape = shape
    elif path == 'block':
        shape = (batch,) + _dims(case) + (steps,)
        i = torch.arange(case['taps'], dtype=torch.float32, device=DEVICE)
        block = torch.nn.Module()
        block.neuron = slayer.neuron.cuba.Neuron(threshold=1.25, current_decay=0.25, voltage_decay=0.03)
        block.delay = slayer.axon.Delay(max_delay=62)
        block.to(DEVICE)
        st.update(x=_spikes(gen, shape, 0.03), taps=(i / 4) * torch.exp(1 - i / 4), block=block)
        block.delay.per_neuron(st['x'])
        block.delay.delay.data = torch.rand(shape[1], generator=gen, device=DEVICE) * 32
        _settled(block.neuron, st['x'])
        st['delay'] = block.delay.delay
        wrt = ['x', 'delay']
        out_shape = shape
    elif path in ('conv', 'dense'):
        neuron = slayer.neuron.cuba.Neuron(threshold=1.25, current_decay=0.25, voltage_decay=0.03)
        if path == 'conv':
            synapse = slayer.synapse.Conv(case['inputs'], case['outputs'], case['kernel'], stride=case['stride'],
                                          padding=case['padding'], pre_hook_fx=neuron.quantize_8bit)
            x = _spikes(gen, (batch, case['inputs'], case['height'], case['width'], steps), 0.05)
            fan_in = case['inputs'] * case['kernel'] ** 2
        else:
            synapse = slayer.synapse.Dense(case['inputs'], case['outputs'], pre_hook_fx=neuron.quantize_8bit)
            x = _spikes(gen, (batch, case['inputs'], steps), 0.03)
            fan_in = case['inputs']
        neuron.to(DEVICE), synapse.to(DEVICE)
        _weights(gen, synapse, 3.0 / math.sqrt(fan_in))
        st.update(x=x, weight=synapse.weight, synapse=synapse, neuron=neuron)
        with torch.no_grad():
            out_shape = neuron(synapse(x)).shape
        wrt = ['x', 'weight']
    elif path == 'decoder':
        pool = slayer.synapse.Pool(2).to(DEVICE)
        up = slayer.synapse.ConvTranspose(case['inputs'], case['outputs'], 4, stride=2, padding=1,
                                          pre_hook_fx=slayer.neuron.cuba.Neuron(1.0, 0.25, 0.25).quantize_8bit).to(DEVICE)
        _weights(gen, up, 3.0 / math.sqrt(case['inputs'] * 4))
        st.update(x=_spikes(gen, (batch, case['inputs'], case['height'], case['width'], steps), 0.05), pool=pool, up=up,
                  weight=up.weight)
        wrt = ['x', 'weight']
        out_shape = (batch, case['outputs'], case['height'], case['width'], steps)
    else:
        n = case['neurons']
        if case['model'] == 'cuba':
            neuron = slayer.neuron.cuba.Neuron(threshold=1.25, current_decay=0.25, voltage_decay=0.25,
                                               persistent_state=True)
            rest = dict(current_state=0.0, voltage_state=0.0)
        else:
            neuron = slayer.neuron.alif.Neuron(threshold=1.25, threshold_step=0.5, current_decay=0.25,
                                               voltage_decay=0.25, threshold_decay=0.25, refractory_decay=0.25,
                                               persistent_state=True)
            rest = dict(current_state=0.0, voltage_state=0.0, threshold_state=1.25, refractory_state=0.0)
        synapse = slayer.synapse.Dense(n, n, pre_hook_fx=neuron.quantize_8bit).to(DEVICE)
        _weights(gen, synapse, 3.6 / math.sqrt(n))
        st.update(x=random(batch, n, steps) * 1.5, weight=synapse.weight, synapse=synapse, neuron=neuron.to(DEVICE),
                  rest={k: torch.full((batch, n), v, device=DEVICE) for k, v in rest.items()})
        wrt = ['x', 'weight']
        out_shape = (batch, n, steps)

    if train:
        st.update(upstream=random(*out_shape), wrt=[st[k].requires_grad_() for k in wrt])
    return st


# ------------------------------------------------------------------------------------------------ one pass
def _forward(st, path):
    """(the tensor gradients come back from, further outputs)."""
    if path == 'dynamics':
        leaky = slayer.neuron.dynamics.leaky_integrator.dynamics
        current = leaky(st['x'], st['current_decay'], st['state'], 64)
        voltage = leaky(current, st['voltage_decay'], st['state'], 64, st['threshold'])
        return slayer.spike.Spike.apply(voltage, st['threshold'], 1.0, 1.0, False, 0, 1), [voltage.detach()]
    if path == 'neuron':
        return st['neuron']((st['x'], st['x_imag']) if 'x_imag' in st else st['x']), []
    if path == 'block':
        return slayer.block.neuron_delay(st['block'], slayer.utils.filter.conv(st['x'], st['taps'], 1)), []
    if path == 'decoder':
        return st['up'](st['pool'](st['x'])), []
    if path == 'recurrent':
        for name, value in st['rest'].items():                # every sequence starts at rest
            setattr(st['neuron'], name, value)
        return slayer.utils.recurrent.custom_recurrent(st['x'], st['neuron'], st['synapse']), []
    return st['neuron'](st['synapse'](st['x'])), []


def run(state):
    path = state['case']['path']
    if not state['case']['train']:
        with torch.no_grad():
            out, more = _forward(state, path)
        return [out] + more
    out, more = _forward(state, path)
    grads = torch.autograd.grad(out, state['wrt'], state['upstream'])
    return [out.detach()] + more + list(grads)


# ------------------------------------------------------------------------------------------------ figures
def work(case):
    """Every operator call of the pass reads its inputs once and writes its results once; what a forward call has to
    leave for its backward call (a state trace) counts once on either side."""
    path, train, steps, batch = case['path'], case['train'], case['steps'], case['batch']
    if path == 'dynamics':
        nt = batch * math.prod(_dims(case)) * steps
        return {'bytes': nt * (60 if train else 24), 'flops': nt * (22 if train else 9)}
    if path == 'neuron':
        nt = batch * math.prod(_dims(case)) * steps
        forward = {'cuba': 8, 'alif': 8, 'rf': 12}[case['model']]
        # training: the trace(s) the surrogate needs, written and read back, the upstream and the input gradient
        both = {'cuba': 24, 'alif': 32, 'rf': 40}[case['model']]
        if case['learn'] and case['model'] == 'cuba':
            both += 8
        return {'bytes': nt * (both if train else forward), 'flops': nt * 30}
    if path == 'block':
        nt = batch * math.prod(_dims(case)) * steps
        return {'bytes': nt * (44 if train else 16), 'flops': nt * ((4 if train else 2) * case['taps'] + 20)}
    if path == 'dense':
        into, out = batch * case['inputs'] * steps, batch * case['outputs'] * steps
        product = 2 * into * case['outputs']
        if not train:
            return {'bytes': 4 * into + 16 * out, 'flops': product}
        return {'bytes': 12 * into + 36 * out, 'flops': 3 * product}
    if path == 'conv':
        ho = (case['height'] + 2 * case['padding'] - case['kernel']) // case['stride'] + 1
        wo = (case['width'] + 2 * case['padding'] - case['kernel']) // case['stride'] + 1
        into = batch * case['inputs'] * case['height'] * case['width'] * steps
        out = batch * case['outputs'] * ho * wo * steps
        product = 2 * out * case['inputs'] * case['kernel'] ** 2
        if not train:
            return {'bytes': 4 * into + 12 * out, 'flops': product}
        return {'bytes': 12 * into + 36 * out, 'flops': 3 * product}
    if path == 'decoder':
        into = batch * case['inputs'] * case['height'] * case['width'] * steps
        out = batch * case['outputs'] * case['height'] * case['width'] * steps
        product = 2 * out * case['inputs'] * 4
        if not train:
            return {'bytes': 6 * into + 4 * out, 'flops': product}
        return {'bytes': 13 * into + 12 * out, 'flops': 3 * product}
    nt = batch * case['neurons'] * steps
    matrix = case['neurons'] ** 2 * 4
    product = 2 * nt * case['neurons']
    trace = 8 if case['model'] == 'alif' else 4
    if not train:
        return {'bytes': 8 * nt + matrix, 'flops': product}
    return {'bytes': nt * (24 + 2 * trace) + 3 * matrix, 'flops': 3 * product}


def tolerance(case):
    """Forward results are fixed-point states and spikes: every bit (the block's depend on the float32 filter in front
    of the neuron).  Gradients are float32 sums: four times what the same pass differs by, on the listed sizes or a
    part of their batch, when its sums are taken in another order (the backward recurrences as scans and step by step,
    the recurrent layer's products by another kernel) or in float64 (the synapses', the filter)."""
    path = case['path']
    if not case['train'] and path != 'block':
        return 'exact'
    if path == 'dynamics':
        return {'rel': 4e-6, 'max': 6e-5}        # 9.2e-7 (a decay gradient), 1.4e-5
    if path == 'neuron':
        # decay gradients cancel to a small part of their terms: 6.2e-6, 1.4e-4; the input's: 5.4e-7, 4.1e-5
        return {'rel': 2.5e-5, 'max': 6e-4} if case['learn'] else {'rel': 2e-6, 'max': 2e-4}
    if path == 'block':
        return {'rel': 1e-6, 'max': 1.5e-5}      # 2.4e-7, 3.2e-6
    if path == 'recurrent':
        return {'rel': 1e-6, 'max': 5e-6}        # 5.6e-8, 1.3e-6; another order in every step of the feedback
    return {'rel': 1.6e-6, 'max': 2.1e-5}        # conv, decoder, dense: 4.0e-7, 5.2e-6
