// tn_apron.hpp -- the interface fields of a label volume laid out for the device's
// queries, and those queries over it.
//
// The reference's layout (Grid::phi) holds 8^3 values per (brick, label): a trilinear
// cell at a brick's upper faces has corners in up to eight bricks, and a third of all
// cells (1 - (7/8)^3) are such. Read as stored, each of those costs up to eight dependent
// lookups (a brick's label list, then its value), and one lane of a wave there makes the
// wave wait for them. Here every (brick, label) slot carries the values of its 9^3
// corners, its own voxels and the layer beyond its upper faces as v2m_phi_vox reads
// them, so that every cell of a brick reads one slot: four pairs of x-neighbours. The
// label list, its count and first slot of a brick share one 64-byte line. Both are laid
// out once per plan or seeding (k_apron, k_brick_rec: 0.23 ms for 256^3 voxels, 44 k
// slots) and the values are bit for bit the ones the stored layout gives; what a slot
// cannot answer (a label the cell's brick does not list, a uniform brick's edge, a cell
// outside the grid) takes the stored layout voxel by voxel, in a loop small enough to be
// inlined. The kernels over it therefore hold no calls and a fraction of the registers:
// the general move pass takes 146 instead of 280, three waves a SIMD instead of one.
// Measured, stored layout -> slots: 2.5 M nodes of a 256^3 volume, general pass 466 ->
// 63 us an iteration, lean interface pass 159 -> 68, k_move_easy 398 -> 278, seeding's
// classification 2.1 -> 0.33 ms; 1.5 M nodes of a probability volume (400 k nodes in the
// general pass), 2.17 -> 0.69 ms, its handed-back nodes 1.08 -> 0.13 ms.
#pragma once

namespace tnd {

constexpr int kApRow = 9, kApPlane = 81;
constexpr int kApSlot = 736;   // 9^3 = 729 values, padded to whole 64-byte lines

// A label volume's grid (gm == 0) with the slots above: the queries below are chosen by
// this type, so that the kernels over it carry no other field mode.
struct PlainField : Field {
    static constexpr bool kPlain = true;
};

template <class F>
__host__ __device__ __forceinline__ F as_field(const Field& f) {
    F r;
    static_cast<Field&>(r) = f;
    return r;
}

// a brick's labels, count and first slot in one line (16 labels, then count and slot)
__global__ __launch_bounds__(256) void k_brick_rec(const int32_t* __restrict__ bl_cnt,
                                                   const uint16_t* __restrict__ bl_lab,
                                                   const int32_t* __restrict__ bl_slot, int nb,
                                                   uint4* __restrict__ rec) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b < nb) {
        const uint4* w = reinterpret_cast<const uint4*>(bl_lab + (size_t)b * kBL);
        rec[(size_t)b * 4] = w[0];
        rec[(size_t)b * 4 + 1] = w[1];
        const int n = bl_cnt[b];
        rec[(size_t)b * 4 + 2] = make_uint4((uint32_t)(n < kBL ? n : kBL), (uint32_t)bl_slot[b], 0u, 0u);
    }
}

// the 9^3 corner values of every slot; a block per brick
__global__ __launch_bounds__(256) void k_apron(Field f, float* __restrict__ ap) {
    const int b = blockIdx.x;
    const int s0 = f.bl_slot[b];
    if (s0 < 0) {
        return;
    }
    const int n = f.bl_cnt[b] < kBL ? f.bl_cnt[b] : kBL;
    const int bi = b % f.nbx, bj = (b / f.nbx) % f.nby, bk = b / (f.nbx * f.nby);
    for (int t = threadIdx.x; t < n * kApSlot; t += 256) {
        const int s = t / kApSlot, e = t % kApSlot;
        float v = 0.0f;
        if (e < kApRow * kApPlane) {
            const int x = e % kApRow, y = (e / kApRow) % kApRow, z = e / kApPlane;
            const int i = 8 * bi + x, j = 8 * bj + y, k = 8 * bk + z;
            if (x < TN_BS && y < TN_BS && z < TN_BS && i < f.nx && j < f.ny && k < f.nz) {
                v = f.phi[(size_t)(s0 + s) * TN_SLOT + (size_t)(x + TN_BS * (y + TN_BS * z))];
            } else {
                v = phi_voxel(f, f.bl_lab[(size_t)b * kBL + s], i, j, k);
            }
        }
        ap[(size_t)(s0 + s) * kApSlot + e] = v;
    }
}

__device__ __forceinline__ BrickList brick_list(const PlainField& f, int b) {
    const uint4* w = f.rec + (size_t)b * 4;
    BrickList r;
    r.lo = w[0];
    r.hi = w[1];
    const uint2 t = *reinterpret_cast<const uint2*>(w + 2);
    r.cnt = (int)t.x;
    r.s0 = (int)t.y;
    return r;
}

// the first of the cell's corners in slot s
__device__ __forceinline__ const float* apron_cell(const PlainField& f, int s, int i0, int j0, int k0) {
    return f.ap + (size_t)s * kApSlot + (size_t)((i0 & 7) + kApRow * (j0 & 7) + kApPlane * (k0 & 7));
}

// (4-byte aligned pairs: a cell starts at any x)
typedef float f32pair __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ void apron_corners(const float* __restrict__ p, float* c) {
    const f32pair r0 = *reinterpret_cast<const f32pair*>(p), r1 = *reinterpret_cast<const f32pair*>(p + kApRow),
                  r2 = *reinterpret_cast<const f32pair*>(p + kApPlane),
                  r3 = *reinterpret_cast<const f32pair*>(p + kApPlane + kApRow);
    c[0] = r0.x;
    c[1] = r0.y;
    c[2] = r1.x;
    c[3] = r1.y;
    c[4] = r2.x;
    c[5] = r2.y;
    c[6] = r3.x;
    c[7] = r3.y;
}

// the corners of phi_l, or of phi_l - phi_m (m >= 0), voxel by voxel from the stored
// layout: a compact loop, so that the rare cells that need it cost the kernels no call
__device__ __forceinline__ void corners_by_voxel(const Field& f, int l, int m, int i0, int j0, int k0, float* c) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        c[e] = 0.0f;
    }
#pragma clang loop unroll(disable)
    for (int q = 0; q < 8; ++q) {
        const int i = step_by(i0, q & 1), j = step_by(j0, (q >> 1) & 1), k = step_by(k0, q >> 2);
        float v = phi_voxel(f, l, i, j, k);
        if (m >= 0) {
            v = v - phi_voxel(f, m, i, j, k);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            c[e] = e == q ? v : c[e];
        }
    }
}

__device__ __forceinline__ void psi_cell_load(const PlainField& f, int a, int b, int i0, int j0, int k0, PsiCell& pc) {
    if (i0 == pc.i0 && j0 == pc.j0 && k0 == pc.k0) {
        return;
    }
    pc.i0 = i0;
    pc.j0 = j0;
    pc.k0 = k0;
    bool slots = false;
    if (in_range(f, i0, j0, k0)) {
        const int bk = brick_at(f, i0, j0, k0);
        if (bk != pc.bk) {
            pc.bk = bk;
            const BrickList bl = brick_list(f, bk);
            int has;
            pc.sa = list_slot(bl, a, &has);
            pc.sb = list_slot(bl, b, &has);
        }
        slots = pc.sa >= 0 && pc.sb >= 0;
    }
    if (slots) {
        float c[8], e[8];
        apron_corners(apron_cell(f, pc.sa, i0, j0, k0), c);
        apron_corners(apron_cell(f, pc.sb, i0, j0, k0), e);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            pc.d[m] = c[m] - e[m];
        }
    } else {
        corners_by_voxel(f, a, b, i0, j0, k0, pc.d);
    }
}

__device__ __forceinline__ float psi_at(const PlainField& f, int a, int b, P3 p, PsiCell& pc) {
    const float u = over_vx(f, p.x), v = over_vy(f, p.y), w = over_vz(f, p.z);
    const int i0 = (int)floorf(u), j0 = (int)floorf(v), k0 = (int)floorf(w);
    psi_cell_load(f, a, b, i0, j0, k0, pc);
    return trilerp(pc.d, u - (float)i0, v - (float)j0, w - (float)k0);
}

__device__ __forceinline__ float4 psi_grad_at(const PlainField& f, int a, int b, P3 p, PsiCell& pc) {
    const float u = over_vx(f, p.x), v = over_vy(f, p.y), w = over_vz(f, p.z);
    const int i0 = (int)floorf(u), j0 = (int)floorf(v), k0 = (int)floorf(w);
    psi_cell_load(f, a, b, i0, j0, k0, pc);
    return trilerp_grad(f, pc.d, u - (float)i0, v - (float)j0, w - (float)k0);
}

__device__ __forceinline__ float4 psi_grad_once(const PlainField& f, int a, int b, P3 p) {
    PsiCell pc;
    psi_cell_init(pc);
    return psi_grad_at(f, a, b, p, pc);
}

__device__ __forceinline__ BrickLabels brick_labels_at(const PlainField& f, P3 p) {
    const int i = (int)floorf(over_vx(f, p.x) + 0.5f), j = (int)floorf(over_vy(f, p.y) + 0.5f),
              k = (int)floorf(over_vz(f, p.z) + 0.5f);
    BrickLabels r;
    if (!in_range(f, i, j, k)) {
        r.b = -1;
        r.n = 1;
        r.list.lo = r.list.hi = make_uint4(0u, 0u, 0u, 0u);
        r.list.cnt = 1;
        r.list.s0 = -1;
        return r;
    }
    r.b = brick_at(f, i, j, k);
    r.list = brick_list(f, r.b);
    r.n = r.list.cnt;
    return r;
}

// The trilinear cell of a point beside the labels of its rounded voxel's brick: in that
// brick the slot of its s-th label is its first slot + s; a cell of the brick below has
// that brick's own list searched.
struct ApronCell {
    int i0, j0, k0;
    float fx, fy, fz;
    bool in, same;     // inside the grid; in the labels' own brick
    BrickList list;    // the cell's brick's list (in)
};

__device__ __forceinline__ ApronCell apron_point(const PlainField& f, P3 p, const BrickLabels& bl) {
    ApronCell c;
    const float u = over_vx(f, p.x), v = over_vy(f, p.y), w = over_vz(f, p.z);
    c.i0 = (int)floorf(u);
    c.j0 = (int)floorf(v);
    c.k0 = (int)floorf(w);
    c.fx = u - (float)c.i0;
    c.fy = v - (float)c.j0;
    c.fz = w - (float)c.k0;
    c.in = in_range(f, c.i0, c.j0, c.k0);
    const int bk = c.in ? brick_at(f, c.i0, c.j0, c.k0) : -1;
    c.same = c.in && bk == bl.b;
    c.list = bl.list;
    if (c.in && !c.same) {
        c.list = brick_list(f, bk);
    }
    return c;
}

// the slot of label l (the s-th of bl; s < 0: any label) at the cell, or -1
__device__ __forceinline__ int apron_slot(const ApronCell& c, int s, int l) {
    if (c.same && s >= 0) {
        return c.list.s0 < 0 ? -1 : c.list.s0 + s;
    }
    int has;
    return c.in ? list_slot(c.list, l, &has) : -1;
}

__device__ __forceinline__ void apron_label_corners(const PlainField& f, const ApronCell& c, int s, int l, float* v) {
    const int sl = apron_slot(c, s, l);
    if (sl >= 0) {
        apron_corners(apron_cell(f, sl, c.i0, c.j0, c.k0), v);
    } else {
        corners_by_voxel(f, l, -1, c.i0, c.j0, c.k0, v);
    }
}

__device__ __forceinline__ float apron_phi(const PlainField& f, const ApronCell& c, int s, int l) {
    float v[8];
    apron_label_corners(f, c, s, l, v);
    return trilerp(v, c.fx, c.fy, c.fz);
}

__device__ __forceinline__ float phi_point(const PlainField& f, int l, P3 p) {
    BrickLabels none;
    none.b = -1;
    return apron_phi(f, apron_point(f, p, none), -1, l);
}

// v2m_label_of (voxmode 0), src/opencl/v2m_seed_body.cl:116-175: (best, second)
__device__ __forceinline__ int2 owner_at(const PlainField& f, P3 p) {
    const BrickLabels bl = brick_labels_at(f, p);
    int best = bl.b < 0 ? 0 : list_label(bl.list, 0), sec = kNoLab;
    if (bl.n == 1) {
        return make_int2(best, kNoLab);
    }
    const ApronCell c = apron_point(f, p, bl);
    float pb = -1.0f, ps = pb;
    for (int s = 0; s < bl.n; ++s) {
        const int l = list_label(bl.list, s);
        const float v = apron_phi(f, c, s, l);
        if (v > pb) {
            ps = pb;
            sec = best;
            pb = v;
            best = l;
        } else if (v > ps) {
            ps = v;
            sec = l;
        }
    }
    return make_int2(best, sec);
}

// The labels ranked two at a time: a mixed brick has at least two, and their corners
// are then in flight together.
__device__ __forceinline__ OwnerPsi owner_psi_at(const PlainField& f, int a, P3 p) {
    OwnerPsi r;
    const BrickLabels bl = brick_labels_at(f, p);
    r.best = bl.b < 0 ? 0 : list_label(bl.list, 0);
    r.sec = kNoLab;
    r.g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (bl.n == 1) {
        return r;
    }
    const ApronCell c = apron_point(f, p, bl);
    float pb = -1.0f, ps = pb;
    float cb[8], cs[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        cb[m] = cs[m] = 0.0f;
    }
    auto rank = [&](int l, const float* v8) {
        const float v = trilerp(v8, c.fx, c.fy, c.fz);
        const bool up = v > pb, mid = !up && v > ps;
        ps = up ? pb : (mid ? v : ps);
        r.sec = up ? r.best : (mid ? l : r.sec);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            cs[m] = up ? cb[m] : (mid ? v8[m] : cs[m]);
            cb[m] = up ? v8[m] : cb[m];
        }
        pb = up ? v : pb;
        r.best = up ? l : r.best;
    };
    for (int s = 0; s < bl.n; s += 2) {
        const int l0 = list_label(bl.list, s), l1 = s + 1 < bl.n ? list_label(bl.list, s + 1) : l0;
        const int s0 = apron_slot(c, s, l0), s1 = s + 1 < bl.n ? apron_slot(c, s + 1, l1) : s0;
        float v0[8], v1[8];
        if (s0 >= 0 && s1 >= 0) {
            apron_corners(apron_cell(f, s0, c.i0, c.j0, c.k0), v0);
            apron_corners(apron_cell(f, s1, c.i0, c.j0, c.k0), v1);
        } else {
            corners_by_voxel(f, l0, -1, c.i0, c.j0, c.k0, v0);
            corners_by_voxel(f, l1, -1, c.i0, c.j0, c.k0, v1);
        }
        rank(l0, v0);
        if (s + 1 < bl.n) {
            rank(l1, v1);
        }
    }
    if (r.best == a && r.sec != kNoLab) {
        float d[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            d[m] = cb[m] - cs[m];
        }
        r.g = trilerp_grad(f, d, c.fx, c.fy, c.fz);
    }
    return r;
}

}  // namespace tnd
