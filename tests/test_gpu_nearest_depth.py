"""ALPHA_BLEND_FIRST_K leaves an instance out of a batch by a depth that none of its fragments is nearer than (nearest_depth).  In discs
far thinner than a pixel and 10^4 to 10^5 times as wide the quadratics of the walk cancel, and a fragment's computed depth can lie well
outside of the Gaussian's own extent: those below were found by evaluating millions of them in 32 bits.  The expected image walks every
instance (the oracle)."""
import numpy as np
import pytest
import torch

from htgs_amd.synthetic import SH_C0, Scene, pinhole
from htgs_amd.torch_bindings import FrameBuffers, RasterizerMode
from util import oracle_render

pytestmark = pytest.mark.gpu

EDGE, FOCAL, K = 512, 200.0, 4

# position, scales, rotation, opacity; the pixel; the depth of the fragment there, and the least one that its extent has room for
THIN = [
    ((-3.87974906, -23.1874142, 23.7906761), (0.000371827336, 37.1827354, 36.8988533), (0.925011575, 0.374729425, -0.0627016649, -0), 0.0500129499, (223, 63), 18.5644, 20.674),
    ((-4.49853849, -0.387633801, 11.1631784), (0.000394668925, 39.4668922, 28.7098961), (0.981590927, 0.0163988657, -0.190290108, -0), 0.050030794, (175, 263), 7.92267, 8.78525),
    ((8.94711208, -8.44185448, 24.6837978), (0.000614797056, 61.4797058, 61.1342735), (0.973401546, 0.157225877, 0.166641608, 0), 0.0514282659, (328, 187), 4.25303, 9.51649),
    ((-0.29767856, 1.93532979, 2.54933953), (4.44575162e-05, 0.444575161, 0.278795093), (0.946846962, -0.317960501, -0.0488057137, -0), 0.0500717163, (232, 412), 2.50641, 2.515),
    ((4.06286478, -1.80827153, 7.73775768), (0.000192635067, 19.2635078, 14.8971539), (0.966179371, 0.104850814, 0.235592335, 0), 0.0501168035, (360, 218), 6.0151, 6.27503),
    ((1.26109743, -0.142068818, 1.25558627), (2.9545572e-05, 2.95455718, 2.04199958), (0.922855079, 0.0431062616, 0.382727563, 0), 0.0501517579, (456, 241), 1.06748, 1.08782),
    ((5.26858282, 4.08581495, 8.34092808), (0.000179652299, 17.965229, 17.6535587), (0.943693161, -0.202737629, 0.261420488, 0), 0.0503223687, (383, 363), 6.10259, 6.11994),
    ((0.848629117, 0.326604724, 1.94039357), (3.17752092e-05, 0.317752093, 0.295261353), (0.976100802, -0.0780732483, 0.202809826, 0), 0.0500286184, (343, 290), 1.89071, 1.91627),
    ((0.225612715, 0.170207232, 1.14556003), (2.32143339e-05, 2.32143331, 1.76621997), (0.99269551, -0.0726619884, 0.0963113457, 0), 0.0500276089, (295, 293), 0.947244, 0.991013),
]


def hidden_scene(position, scales, rotation, opacity, pixel, depth, extent):
    """64 black discs across the view, the first four of them between the fragment and where its extent begins: they fill the cores of the
    tile before the Gaussian, which is white and the last by index, is looked at."""
    between = 0.5 * (depth + extent)
    z = torch.cat([between * (1.0 + 1e-5 * torch.arange(4)), (1.2 + 0.005 * torch.arange(60)) * max(extent, between)])
    x, y = [(v + 0.5 - EDGE / 2) / FOCAL for v in pixel]
    discs = torch.stack([x * z, y * z, z], 1)
    n = 65
    rotations = torch.zeros(n, 4)
    rotations[:, 0] = 1.0
    rotations[-1] = torch.tensor(rotation)
    opacities = torch.full((n, 1), 0.5)
    opacities[-1] = opacity
    sh_0 = torch.full((n, 1, 3), -0.5 / SH_C0)
    sh_0[-1] = 0.5 / SH_C0
    M, VPM, cam = pinhole(EDGE, EDGE, FOCAL, FOCAL, EDGE / 2, EDGE / 2, 0.1, 100.0)
    return Scene("thin", torch.cat([discs, torch.tensor([position])]), torch.cat([torch.stack([0.3 * z, 0.3 * z, 1e-3 * z], 1), torch.tensor([scales])]), rotations,
                 opacities, sh_0, torch.zeros(n, 0, 3), M, VPM, cam, EDGE, EDGE, 0.1, 100.0, 1, K)


@pytest.mark.parametrize("waves", [1, 2])
@pytest.mark.parametrize("which", range(len(THIN)))
def test_fragments_outside_of_the_extent(cuda, which, waves):
    print(f"case which={which} waves={waves}", flush=True)
    scene = hidden_scene(*THIN[which])
    x, y = THIN[which][4]
    want = oracle_render(scene, 1, K)
    assert want["image"][:, y, x].min() > 0.04                 # (its alpha at the pixel, 1/20, times white: it is the nearest there)
    sg = scene.to(cuda)
    for train in (False, True):
        fb = FrameBuffers(*sg.gaussians(), sg.settings(RasterizerMode(1), K), True, False, train=train, waves_per_tile=waves)
        image = fb.run_forward() if train else fb.run()[0]
        assert np.abs(image.cpu().numpy() - want["image"]).max() <= 1e-4
