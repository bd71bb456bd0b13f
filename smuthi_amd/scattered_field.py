"""Plane wave expansion of the scattered field with the particle sum on the
GPU (postprocessing/scattered_field.py:13-150): for every layer of the
scatterers, the outgoing SWE -> PWE conversion
(fields/transformations.py:133-226) of all particles is summed in one
libsmh launch (smh_pwe_assemble); the direct part and the layer response
(layers.py:141-191) are combined on the host.
"""
import copy
import ctypes

import numpy as np

from . import _lib
from . import cuda as cu
from . import fields as flds
from . import layers as lay
from . import special as sf
from .expansions import PiecewiseFieldExpansion, PlaneWaveExpansion, SphericalWaveSum


def _coefficients(particle):
    swe = particle.scattered_field
    if swe is None:
        raise ValueError('particle has no scattered field (solve the linear system first)')
    return np.asarray(getattr(swe, 'coefficients', swe), dtype=complex)


class _Scatterers:
    """The particles of one layer as arrays: positions, coefficients on common cut-offs l_max, m_max."""

    def __init__(self, particles, xyz):
        self.xyz = np.ascontiguousarray(xyz)
        self.l_max = max(p.l_max for p in particles)
        self.m_max = max(p.m_max for p in particles)
        self.coefficients = np.zeros((len(particles), flds.blocksize(self.l_max, self.m_max)), complex)
        # particles grouped by their own (l_max, m_max): one index map and one array copy per group
        groups = {}
        for i, p in enumerate(particles):
            groups.setdefault((p.l_max, p.m_max), []).append(i)
        for (lp, mp), idx in groups.items():
            dst = [flds.multi_to_single_index(tau, l, m, self.l_max, self.m_max)
                   for tau in range(2) for l in range(1, lp + 1) for m in range(-min(l, mp), min(l, mp) + 1)]
            src = [flds.multi_to_single_index(tau, l, m, lp, mp)
                   for tau in range(2) for l in range(1, lp + 1) for m in range(-min(l, mp), min(l, mp) + 1)]
            block = np.stack([_coefficients(particles[i]) for i in idx])
            self.coefficients[np.asarray(idx)[:, None], np.asarray(dst)[None, :]] = block[:, src]


def _layer_numbers(layer_system, z):
    """layer_system.layer_number of every height. One search finds them all where that is LayerSystem's own; a
    layer system of another class, or with a layer_number of its own, is asked height by height."""
    ask = layer_system.layer_number
    if (isinstance(layer_system, lay.LayerSystem) and getattr(ask, '__func__', None) is lay.LayerSystem.layer_number
            and ask.__self__ is layer_system):
        return layer_system.layer_numbers(z)
    return np.array([ask(h) for h in z])


def _by_layer(particle_list, layer_system):
    """[(layer, its particles, their positions)] in the order of the layers."""
    particle_list = list(particle_list)
    if not particle_list:
        return []
    xyz = np.array([p.position for p in particle_list], dtype=np.float64)
    layers = _layer_numbers(layer_system, xyz[:, 2])
    out = []
    for i in np.unique(layers):
        idx = np.flatnonzero(layers == i)
        out.append((int(i), [particle_list[j] for j in idx], xyz[idx]))
    return out


def _assemble(vacuum_wavelength, parts, layer_system, i_swe, k_parallel, azimuthal_angles, precision):
    """(g_up, g_dn), each [2, n_k, n_a], of the _Scatterers of layer i_swe at reference [0, 0, z_ref(i_swe)]."""
    om = flds.angular_frequency(vacuum_wavelength)
    k = complex(om * layer_system.refractive_indices[i_swe])
    l_max, m_max, xyz, coef = parts.l_max, parts.m_max, parts.xyz, parts.coefficients
    kp = np.ascontiguousarray(np.array(k_parallel, ndmin=1), dtype=complex)
    kz = flds.k_z(k_parallel=kp, k=k).astype(complex)
    # B_{n,pol}(+-kz/k, kappa/k) / (2 pi kz k): btab[k][dir][pol][n]
    bu = sf.transformation_arrays(l_max, m_max, kz / k, kp / k, False)
    bd = sf.transformation_arrays(l_max, m_max, -kz / k, kp / k, False)
    den = 2 * np.pi * kz * k
    btab = np.ascontiguousarray(np.stack([bu, bd]).transpose(3, 0, 1, 2) / den[:, None, None, None])
    al = np.ascontiguousarray(np.array(azimuthal_angles, ndmin=1), dtype=np.float64)
    g = np.zeros((2, 2, len(kp), len(al)), complex)
    ms = ctypes.c_double()
    prec = _lib.FP64 if precision in ('double', 'double precision') else _lib.FP32
    _lib.check(_lib.load().smh_pwe_assemble(cu.context(), len(xyz), _lib.dptr(xyz), l_max, m_max, _lib.dptr(coef),
                                             float(layer_system.reference_z(i_swe)), len(kp), _lib.dptr(kp),
                                             _lib.dptr(np.ascontiguousarray(kz)), _lib.dptr(btab), len(al),
                                             _lib.dptr(al), _lib.dptr(g), prec, ctypes.byref(ms)),
               cu.context(), 'smh_pwe_assemble')
    return g[0], g[1], k, kp, al, ms.value


def scattered_field_pwe(vacuum_wavelength, particle_list, layer_system, layer_number, k_parallel='default',
                        azimuthal_angles='default', include_direct=True, include_layer_response=True,
                        precision='single'):
    """(upgoing, downgoing) PlaneWaveExpansion of the scattered field in layer_number
    (postprocessing/scattered_field.py:80-150)."""
    return _scattered_field_pwe(vacuum_wavelength, _by_layer(particle_list, layer_system), {}, layer_system,
                                layer_number, k_parallel, azimuthal_angles, include_direct, include_layer_response,
                                precision, (0, 1))


def _scattered_field_pwe(vacuum_wavelength, by_layer, scatterers, layer_system, layer_number, k_parallel,
                         azimuthal_angles, include_direct, include_layer_response, precision, directions):
    """scattered_field_pwe for particles grouped by _by_layer. Only the expansions of the given directions
    (0 up, 1 down) are filled; scatterers keeps the layers' arrays between calls of one far field.

    The sums run in place: the expansions of a layer share their grids, and its response matrices serve both
    directions of the source (1000 spheres, 91 x 361 directions in each half space: 11.3 ms per far field when
    every term was an expansion of its own, added with the checks of PlaneWaveExpansion.__add__, and every
    particle's layer searched for by itself)."""
    if isinstance(k_parallel, str) and k_parallel == 'default':
        k_parallel = flds.default_Sommerfeld_k_parallel_array
    if isinstance(azimuthal_angles, str) and azimuthal_angles == 'default':
        azimuthal_angles = flds.default_azimuthal_angles
    om = flds.angular_frequency(vacuum_wavelength)
    k = om * layer_system.refractive_indices[layer_number]
    z = layer_system.reference_z(layer_number)
    vb = (layer_system.lower_zlimit(layer_number), layer_system.upper_zlimit(layer_number))
    out = [PlaneWaveExpansion(k, k_parallel, azimuthal_angles, kind, [0, 0, z], vb[0], vb[1])
           for kind in ('upgoing', 'downgoing')]
    scattered_field_pwe.last_kernel_ms = 0.0
    for i_swe, particles, xyz in by_layer:
        direct = i_swe == layer_number and include_direct
        if not (direct or include_layer_response):
            continue
        if i_swe not in scatterers:
            scatterers[i_swe] = _Scatterers(particles, xyz)
        *g, k_swe, kp, al, ms = _assemble(vacuum_wavelength, scatterers[i_swe], layer_system, i_swe, k_parallel,
                                          azimuthal_angles, precision)
        scattered_field_pwe.last_kernel_ms += ms
        # the terms' common grids (the assembly's), wavenumber and reference point, as PlaneWaveExpansion.__add__
        # checks them
        n = layer_system.refractive_indices
        term = copy.copy(out[0])
        term.k, term.k_parallel, term.azimuthal_angles = k_swe / n[i_swe] * n[layer_number], kp, al
        term.reference_point = list(out[0].reference_point)
        if not out[0].compatible(term):
            raise ValueError('Plane wave expansion are inconsistent.')
        if direct:
            out[0].lower_z, out[1].upper_z = max(vb[0], xyz[:, 2].max()), min(vb[1], xyz[:, 2].min())
            for d in directions:
                out[d].coefficients += g[d]
        if include_layer_response:
            for pol in range(2):
                L = lay.layersystem_response_matrix(pol, layer_system.thicknesses, layer_system.refractive_indices,
                                                    kp, k_swe / layer_system.refractive_indices[i_swe], i_swe,
                                                    layer_number)
                for d in directions:
                    out[d].coefficients[pol] += L[d, 0][:, None] * g[0][pol] + L[d, 1][:, None] * g[1][pol]
    return tuple(out)


def scattered_field_piecewise_expansion(vacuum_wavelength, particle_list, layer_system, k_parallel='default',
                                        azimuthal_angles='default', layer_numbers=None, precision='single'):
    """Scattered field as a PiecewiseFieldExpansion
    (postprocessing/scattered_field.py:13-77): per layer the layer-mediated
    upgoing (not in the bottom layer) and downgoing (not in the top layer)
    plane wave expansions, plus the direct field, the particles' outgoing
    spherical wave expansions, summed on the GPU per layer
    (expansions.SphericalWaveSum); points inside a particle get no field."""
    if layer_numbers is None:
        layer_numbers = range(layer_system.number_of_layers())
    nl = layer_system.number_of_layers()
    particle_list = list(particle_list)
    sfld = PiecewiseFieldExpansion()
    for i in layer_numbers:
        up, dn = scattered_field_pwe(vacuum_wavelength, particle_list, layer_system, i, k_parallel, azimuthal_angles,
                                     include_direct=False, include_layer_response=True, precision=precision)
        if i > 0:
            sfld.expansion_list.append(up)
        if i < nl - 1:
            sfld.expansion_list.append(dn)
    for i, parts, _ in _by_layer(particle_list, layer_system):
        k = flds.angular_frequency(vacuum_wavelength) * layer_system.refractive_indices[i]
        sfld.expansion_list.append(SphericalWaveSum(k, parts, layer_system.lower_zlimit(i),
                                                    layer_system.upper_zlimit(i)))
    for p in particle_list:
        sfld.validity_conditions.append(p.is_outside)
    return sfld
