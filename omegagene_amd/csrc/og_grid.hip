// og_grid.hip -- device build of the 8-atom-cell grid and the cell-pair list.
//
// Bit-exact integer work: column binning, column order, in-column z order,
// dummy padding, uniform-z bins, cell-pair enumeration order and the 64-bit
// exclusion masks reproduce MiniCell (src/celeste/core/MiniCell.cpp) on the
// same FP64 coordinates.  This file is compiled with -ffp-contract=off and
// correctly rounded float division so every float expression rounds where
// the reference host build rounds it.
#include "og_internal.h"

// ---------------------------------------------------------------- clear --
// Empties thread t's share (every n-th) of the uniform-z bin table.
__device__ __forceinline__ void og_clear_bins(const og_dev_sys &s, const int t, const int n) {
    const int n_bins = (s.n_columns + 1) * s.n_uni_z;
    for (int k = t; k < n_bins; k += n) {
        s.u2c_min[k] = OG_EMPTY_BIN;
        s.u2c_max[k] = -1;
    }
}
// The bin table of the reference call points (an engine's rebuild empties it
// in k_grid_bin).
__global__ void __launch_bounds__(OG_THREADS) k_grid_clear(const og_dev_sys *__restrict__ S,
                                                           const int2 *__restrict__ map) {
    const int2        bm = map[blockIdx.x];
    const og_dev_sys &s  = S[bm.x];
    if (og_rebuild_skip(s)) return;
    og_clear_bins(s, blockIdx.x * OG_THREADS + threadIdx.x, gridDim.x * OG_THREADS);
    // overflow flags stay set until the host has read them (check_flags), so a
    // failed rebuild inside a multi-step graph is never hidden by a later one
}

// ------------------------------------------------------------------ bin --
// MiniCell::set_atoms_into_grid_xy binning (MiniCell.cpp:316-359):
//   float x = crd - lb (double subtraction rounded to float), periodic wrap
//   in float, column = floor(x / L_cell) with IEEE float division.
// Wave-aggregated counter add: lanes with the same key share one atomic
// (atoms in input order are mostly spatial neighbours, so a wave touches a
// few columns).  Returns the old counter value plus the lane's rank among
// the lanes of its key, i.e. what a per-lane atomicAdd(ctr + key, 1) could
// have returned.  The keys' atomics go out together: one after the other, a
// wave of chain atoms (ten columns) waited ten round trips (the scatter of
// 4,230 atoms 10.5 us, now 4.1).
__device__ __forceinline__ int og_wave_count_add(int *ctr, int key, bool active) {
    const int lane   = threadIdx.x & 63;
    uint64_t  todo   = __ballot(active);
    int       leader = lane, rank = 0, count = 0;
    while (todo) {
        const int      l    = __builtin_ctzll(todo);
        const int      lkey = __builtin_amdgcn_readlane(key, l);
        const uint64_t m    = __ballot(active && key == lkey) & todo;
        if ((m >> lane) & 1ull) {
            leader = l;
            rank   = __builtin_popcountll(m & ((1ull << lane) - 1ull));
            count  = __builtin_popcountll(m);
        }
        todo &= ~m;
    }
    int base = 0;
    if (active && leader == lane) base = atomicAdd(ctr + key, count);
    return __shfl(base, leader, 64) + rank;
}

// ----------------------------------------------------------------- scan --
// MiniCell::set_idx_xy_head (MiniCell.cpp:785-861): cells per column,
// exclusive scan to head cell/atom, -1 heads for empty columns.  By the last
// block of the binning, which reads the counts of all blocks (a launch of its
// own took 4 us and the gap before it).
__device__ __forceinline__ void og_scan_columns(const og_dev_sys &s) {
    const int nc  = s.n_columns;
    const int per = (nc + OG_THREADS - 1) / OG_THREADS;
    const int k0  = threadIdx.x * per, k1 = min(k0 + per, nc);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __shared__ int wsum[OG_THREADS / 64], big;
    if (threadIdx.x == 0) big = 0;
    auto count = [&](int k) {
        return __hip_atomic_load(&s.n_atoms_col[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    // read with the counts; flagged by the binning (or before it): there is no grid to lay out
    const int flags = __hip_atomic_load(&s.cnt->flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int local = 0, mx = 0;
#pragma unroll 4
    for (int k = k0; k < k1; k++) {
        const int n = count(k);
        local += (n + OG_NAC - 1) / OG_NAC;
        mx = max(mx, n);
    }
    if (flags & OG_F_FATAL) return;
    int incl = local;
    for (int off = 1; off < 64; off <<= 1) {
        const int v = __shfl_up(incl, off, 64);
        if (lane >= off) incl += v;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    if (mx > OG_SORT_CAP) atomicOr(&big, 1);
    __syncthreads();
    int cell = incl - local;
    for (int q = 0; q < w; q++) cell += wsum[q];
#pragma unroll 4
    for (int k = k0; k < k1; k++) {
        const int n  = count(k);
        const int nz = (n + OG_NAC - 1) / OG_NAC;
        s.n_cells_z[k] = nz;
        s.head_cell[k] = n ? cell : -1;
        s.head_atom[k] = n ? cell * OG_NAC : -1;
        s.col_fill[k]  = 0;
        cell += nz;
    }
    if (threadIdx.x == OG_THREADS - 1) {
        int total = cell;
        s.head_cell[nc] = total;
        s.head_atom[nc] = total * OG_NAC;
        int fl = 0;
        if (total > s.cap_cells) fl |= OG_F_CELL_OVERFLOW;
        if (big) fl |= OG_F_COL_OVERFLOW;
        if (fl) {
            atomicOr(&s.cnt->flags, fl);
            total = 0;  // nothing downstream runs on a grid that does not fit
        }
        s.cnt->n_cells = total;
    }
}

// point: a single-point call's rebuild, whatever the step; the last block
// leaves the call's requests for the kernels after it.
__global__ void __launch_bounds__(OG_THREADS) k_grid_bin(const og_dev_sys *__restrict__ S,
                                                         const int2 *__restrict__ map, const int point) {
    const int2        bm = map[blockIdx.x];
    const og_dev_sys &s  = S[bm.x];
    // A launch raises flags itself (non-finite atoms), which the waves of a block may read differently: a wave that
    // finds one does no work, but every block arrives, and the scan reads the flags when all are raised.
    if (s.cnt->step >= s.cnt->step_end || !(point || og_rebuild_due(s))) return;
    const bool        run = (s.cnt->flags & OG_F_FATAL) == 0;
    const int         i  = bm.y * OG_THREADS + threadIdx.x;
    const bool        in = run && i < s.n_atoms;
    if (run) og_clear_bins(s, i, s.n_atom_blocks * OG_THREADS);  // read by the last rebuild only, filled by the sort
    int  c[2] = {0, 0};
    bool bad = false;
    if (in) {
        for (int d = 0; d < 2; d++) {
            const double cd = s.crd[3 * i + d];
            if (!(cd == cd) || cd > 1e30 || cd < -1e30) {
                bad = true;
                c[d] = 0;
                continue;
            }
            if (cd > (double)s.ub[d] || cd < (double)s.lb[d]) atomicOr(&s.cnt->flags, OG_F_OUTSIDE_BOX);
            float x = (float)(cd - (double)s.lb[d]);
            if (x < -4.0f * s.L[d] || x >= 5.0f * s.L[d]) {  // far outside: flag instead of looping
                atomicOr(&s.cnt->flags, OG_F_OUTSIDE_BOX);
                x = 0.0f;
            }
            while (x < 0.0f) x += s.L[d];
            while (x >= s.L[d]) x -= s.L[d];
            int k = (int)floorf(x / s.L_cell[d]);
            const int n = d == 0 ? s.nx : s.ny;
            while (k < 0) k += n;
            while (k >= n) k -= n;
            c[d] = k;
        }
        const double z = s.crd[3 * i + 2];
        if (!(z == z) || z > 1e30 || z < -1e30) bad = true;
        if (bad) atomicOr(&s.cnt->flags, OG_F_NAN);
        const int col    = c[0] + c[1] * s.nx;
        s.col_of_atom[i] = col;
        s.zkey[i]        = og_float_key(bad ? 0.0f : (float)z);
    }
    og_wave_count_add(s.n_atoms_col, c[0] + c[1] * s.nx, in);
    if (!og_last_block_of(s.sync, bm.y, s.n_atom_blocks)) return;
    if (point && threadIdx.x == 0) og_request_point(s.cnt, 1);
    og_scan_columns(s);
}

// -------------------------------------------------------------- scatter --
__global__ void __launch_bounds__(OG_THREADS) k_grid_scatter(const og_dev_sys *__restrict__ S,
                                                             const int2 *__restrict__ map) {
    const int2        bm = map[blockIdx.x];
    const og_dev_sys &s  = S[bm.x];
    if (og_rebuild_skip(s)) return;
    const int         i  = bm.y * OG_THREADS + threadIdx.x;
    if (s.cnt->n_cells == 0) return;
    const bool in   = i < s.n_atoms;
    const int  col  = in ? s.col_of_atom[i] : 0;
    const int  slot = og_wave_count_add(s.col_fill, col, in);
    if (in) s.tmp_ids[s.head_atom[col] + slot] = i;
}

// ----------------------------------------------------------------- sort --
// One block per column.  Ascending float z with the atom id as tie-break
// (the reference Hoare quicksort, MiniCell.cpp:636-691, orders distinct z
// identically; exact float ties inside a column are the only difference),
// then padding to a multiple of 8 with copies of the last real atom
// (MiniCell.cpp:574-580), grid-order coordinates rounded through float
// (MiniCell.cpp:414-415), cell z extents and uniform-z bins
// (MiniCell.cpp:884-936).
//
// A column of at most a block's threads (any at liquid density in a box below
// 150 A) has an atom per thread: it loads its atom while it counts the smaller
// keys (its place), and leaves its z in LDS for the cells.  A longer column is
// sorted in LDS by a bitonic network.  The kernel is a chain of memory round
// trips; the count takes 3 cycles per key and wave against the network's 28
// barriers for 128 atoms (4,230 atoms 10.0 -> 6.2 us).
struct og_slot_atom {
    float x, y, z, q;
    int   type, comp;
};
__device__ __forceinline__ og_slot_atom og_load_slot_atom(const og_dev_sys &s, const int id) {
    return og_slot_atom{(float)s.crd[3 * id], (float)s.crd[3 * id + 1], (float)s.crd[3 * id + 2],
                        s.charge[id], s.atom_type[id], s.comp[id]};
}
// id < 0: a dummy at atom a's place
__device__ __forceinline__ void og_store_slot(const og_dev_sys &s, const int slot, const int id,
                                              const og_slot_atom &a) {
    s.atomids[slot]      = id;
    s.gcrd[3 * slot]     = (double)a.x;
    s.gcrd[3 * slot + 1] = (double)a.y;
    s.gcrd[3 * slot + 2] = (double)a.z;
    s.gxyzq[slot]        = make_float4(a.x, a.y, a.z, id >= 0 ? a.q : 0.0f);
    s.gtype[slot]        = id >= 0 ? a.type : 0;
    s.gcomp[slot]        = id >= 0 ? a.comp : -1;
    if (id >= 0) s.rev[id] = slot;
}

__device__ void og_column_cells(const og_dev_sys &s, int col, int nz, const float *z);

__global__ void __launch_bounds__(OG_THREADS, 8) k_grid_sort(const og_dev_sys *__restrict__ S,
                                                          const int2 *__restrict__ map) {
    const int2        bm  = map[blockIdx.x];
    const og_dev_sys &s   = S[bm.x];
    if (og_rebuild_skip(s)) return;
    const int         col = bm.y;
    __shared__ uint64_t keys[OG_SORT_CAP];
    __shared__ float    zs[OG_THREADS + OG_NAC];
    const int n = s.n_atoms_col[col], nz = s.n_cells_z[col], base = s.head_atom[col];
    if (s.cnt->n_cells == 0) return;
    if (n == 0) return;
    const int tid = threadIdx.x;
    if (n <= OG_THREADS) {
        const int    id = tid < n ? s.tmp_ids[base + tid] : 0;
        og_slot_atom a{};
        uint64_t     key = ~0ull;
        if (tid < n) {
            key = ((uint64_t)s.zkey[id] << 32) | (uint32_t)id;
            a   = og_load_slot_atom(s, id);
        }
        keys[tid] = key;  // past the column: above every key, as far as the unrolled count reads
        __syncthreads();
        if (tid == 0) s.n_atoms_col[col] = 0;  // the next rebuild's binning counts from zero
        if (tid < n) {
            int rank = 0;
            for (int k = 0; k < n; k += 8)
#pragma unroll
                for (int j = 0; j < 8; j++) rank += keys[k + j] < key ? 1 : 0;
            og_store_slot(s, base + rank, id, a);
            zs[rank] = a.z;
            if (rank == n - 1)
                for (int t = n; t < nz * OG_NAC; t++) {
                    og_store_slot(s, base + t, -1, a);
                    zs[t] = a.z;
                }
        }
        __syncthreads();
        og_column_cells(s, col, nz, zs);
        return;
    }
    int P = 1;
    while (P < n) P <<= 1;
    for (int t = tid; t < P; t += OG_THREADS) {
        if (t < n) {
            const int id = s.tmp_ids[base + t];
            keys[t]      = ((uint64_t)s.zkey[id] << 32) | (uint32_t)id;
        } else {
            keys[t] = ~0ull;
        }
    }
    __syncthreads();
    if (tid == 0) s.n_atoms_col[col] = 0;
    for (int k = 2; k <= P; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = tid; t < P; t += OG_THREADS) {
                const int u = t ^ j;
                if (u > t) {
                    const uint64_t a = keys[t], b = keys[u];
                    const bool     up = (t & k) == 0;
                    if ((a > b) == up) {
                        keys[t] = b;
                        keys[u] = a;
                    }
                }
            }
            __syncthreads();
        }
    }
    const int last = (int)(keys[n - 1] & 0xffffffffu);
    for (int t = tid; t < nz * OG_NAC; t += OG_THREADS) {
        const int id = t < n ? (int)(keys[t] & 0xffffffffu) : -1;
        og_store_slot(s, base + t, id, og_load_slot_atom(s, t < n ? id : last));
    }
    __syncthreads();
    og_column_cells(s, col, nz, nullptr);
}

// Cells of one grid column from grid-order coordinates: cell -> column and z
// index, z extents from the first and last slot of each cell (dummies copy
// the last real atom, so the last slot holds the top), and the uniform-z bins
// the cell overlaps (MiniCell::set_uniform_grid, MiniCell.cpp:884-936).
// Called by one block per column after the column's slots are written; z: the
// slots' z in LDS, or null.
__device__ void og_column_cells(const og_dev_sys &s, int col, int nz, const float *z) {
    const int hc = s.head_cell[col];
    for (int c = threadIdx.x; c < nz; c += blockDim.x) {
        const int   cell = hc + c;
        const float zmin = z ? z[c * OG_NAC] : (float)s.gcrd[3 * (cell * OG_NAC) + 2];
        const float zmax = z ? z[c * OG_NAC + OG_NAC - 1] : (float)s.gcrd[3 * (cell * OG_NAC + OG_NAC - 1) + 2];
        s.cell_col[cell]  = col;
        s.cell_z[cell]    = c;
        s.cell_zmin[cell] = zmin;
        s.cell_zmax[cell] = zmax;
        const float a = zmin - s.lb[2];
        const float b = zmax - s.lb[2];
        // (int) truncation as MiniCell.cpp:912-913; the clamp only guards
        // coordinates outside the box (the reference indexes out of bounds there)
        const int u0 = min(max((int)(a / s.L_z_uni), 0), s.n_uni_z);
        const int u1 = min(max((int)(b / s.L_z_uni), u0), s.n_uni_z);
        s.cell_u0[cell] = u0;
        s.cell_u1[cell] = u1;
        for (int u = u0; u <= u1; u++) {
            // uni id = x*n_uni_z + y*n_uni_z*nx + z  (MiniCell.cpp:1596-1598); a top that
            // rounds onto the upper face spills into the next column's first bin, as there.
            const int bin = col * s.n_uni_z + u;
            atomicMin(&s.u2c_min[bin], c);
            atomicMax(&s.u2c_max[bin], c);
        }
    }
}

// Cell tables of a grid built on the host (the reference call points, where
// MiniCell sorts the atoms and uploads atomids, column heads and float
// coordinates): one block per column.
__global__ void __launch_bounds__(OG_THREADS) k_cells_from_grid(const og_dev_sys *__restrict__ S,
                                                                const int2 *__restrict__ map) {
    const int2        bm  = map[blockIdx.x];
    const og_dev_sys &s   = S[bm.x];
    if (og_rebuild_skip(s)) return;
    const int         col = bm.y;
    if (s.head_cell[col] < 0) return;
    og_column_cells(s, col, s.n_cells_z[col], nullptr);
}

// ---------------------------------------------------------- enumeration --
// MiniCell::enumerate_cell_pairs (MiniCell.cpp:938-1149) for one cell1 per
// wave: lane k takes neighbour column k in the reference loop order
// (dx outer, dy inner), walks the three z images and the candidate cells in
// ascending id: the lanes' ranges, one after the other, are the CPU list order.
__device__ __forceinline__ bool og_valid_pair(int c1, int c2) {
    // MiniCell::check_valid_pair (MiniCell.cpp:1150-1160)
    const bool o1 = (c1 & 1) != 0, o2 = (c2 & 1) != 0;
    if (o1) return !((c2 < c1 && !o2) || (c2 > c1 && o2));
    return !((c2 < c1 && o2) || (c2 > c1 && !o2));
}

// Squared z gap between cell2 [z2b, z2t] (image-shifted) and cell1 [z1b, z1t]
// (MiniCell.cpp:1095-1104)
__device__ __forceinline__ float og_zgap2(float z2t, float z2b, float z1b, float z1t) {
    float d2;
    if (z2t < z1b) {
        d2 = z1b - z2t;
        d2 = d2 * d2;
    } else if (z2b > z1t) {
        d2 = z2b - z1t;
        d2 = d2 * d2;
    } else {
        d2 = 0.0f;
    }
    return d2;
}

// MODE 1: count the cell's pairs and stage them (cell2 | image << 24, list
// order) in cp_stage[c1 * OG_ENUM_STAGE ...] as far as they fit;
// MODE 2: write them at p0 (cells whose pairs did not fit).
// Bound by its instructions and gathered loads: with the candidates of a
// column walked by its lane (25 of 64 lanes, 13 steps) it took 148 us at
// 450,000 atoms, 60 for sixteen walkers, 33 at 99,200 atoms; a lane per
// candidate 105, 53 and 29.  Reading a lane's bins eight at a time is slower
// (119, 61 and 31): most windows are five bins.
// LDS written by the wave's lanes is visible to the others after it
__device__ __forceinline__ void og_wave_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}
struct og_enum_lds {  // of one wave
    int4 at[64];    // by lane (neighbour column): candidates before its own, first cell per z image
    int3 run[64];   // cells in images 0 and 1, (x, y) distance squared
    int  mark[65];  // candidate of a chunk -> 1 + the lane whose candidates start there (64: of no chunk)
};
template <int MODE>
__device__ void og_enum_cell(const og_dev_sys &s, og_enum_lds &T, int c1, int p0, int *out_count) {
    const int lane  = threadIdx.x & 63;
    const int col1  = s.cell_col[c1];
    const int x1    = col1 % s.nx, y1 = col1 / s.nx;
    const float z1b = s.cell_zmin[c1], z1t = s.cell_zmax[c1];
    const int   u0  = s.cell_u0[c1], u1 = s.cell_u1[c1];
    const int   wy  = 2 * s.nny + 1;
    const int   ncand = (2 * s.nnx + 1) * wy;
    const int   nuz = s.n_uni_z;
    // z-bin windows per image (MiniCell.cpp:1014-1038)
    int fz[3], lz[3];
    int tf = u0 - 2;
    if (tf < 0) {
        fz[0] = nuz + tf;
        lz[0] = nuz - 1;
        tf    = 0;
    } else {
        fz[0] = lz[0] = -1;
    }
    fz[1]  = tf;
    int tl = u1 + 2;
    if (tl >= nuz) {
        fz[2] = 0;
        lz[2] = tl - nuz;
        lz[1] = nuz - 1;
    } else {
        fz[2] = lz[2] = -1;
        lz[1]         = tl;
    }
    int pos = MODE == 2 ? p0 : 0;  // of the next pair kept
    for (int r0 = 0; r0 < ncand; r0 += 64) {
        const int k     = r0 + lane;
        int       c2lo[3], c2hi[3];
        float     dd01  = 0.0f;
        int       imgxy = 0;
        for (int ii = 0; ii < 3; ii++) c2lo[ii] = 0, c2hi[ii] = -1;
        if (k < ncand) {
            const int dx = k / wy - s.nnx, dy = k % wy - s.nny;
            int       rx = x1 + dx, ry = y1 + dy, cx = rx, cy = ry;
            if (rx < 0) {
                cx = s.nx + rx;
                imgxy |= 1;
            } else if (rx >= s.nx) {
                cx = rx - s.nx;
                imgxy |= 2;
            }
            if (ry < 0) {
                cy = s.ny + ry;
                imgxy |= 4;
            } else if (ry >= s.ny) {
                cy = ry - s.ny;
                imgxy |= 8;
            }
            float d0 = dx > 0 ? (float)(dx - 1) * s.L_cell[0] : dx < 0 ? (float)(dx + 1) * s.L_cell[0] : 0.0f;
            float d1 = dy > 0 ? (float)(dy - 1) * s.L_cell[1] : dy < 0 ? (float)(dy + 1) * s.L_cell[1] : 0.0f;
            d0        = d0 * d0;
            d1        = d1 * d1;
            dd01      = d0 + d1;
            const int col2  = cx + cy * s.nx;
            const int head2 = s.head_cell[col2];
            for (int ii = 0; ii < 3; ii++) {
                if (fz[ii] < 0 || head2 < 0) continue;
                int fu = col2 * nuz + fz[ii], lu = col2 * nuz + lz[ii];
                int f = -1, l = -1;
                if (s.gap_bug) {
                    // stop at the first empty bin after a non-empty one (MiniCell.cpp:1063-1077)
                    int stg = 0;
                    for (int u = fu; u <= lu; u++) {
                        const bool full = s.u2c_min[u] != OG_EMPTY_BIN;
                        if (stg == 0 && full) {
                            stg = 1;
                            f   = u;
                            l   = lu;
                        } else if (stg == 1 && !full) {
                            l = u - 1;
                            break;
                        }
                    }
                } else {
                    for (int u = fu; u <= lu; u++)
                        if (s.u2c_min[u] != OG_EMPTY_BIN) {
                            if (f < 0) f = u;
                            l = u;
                        }
                }
                if (f < 0) continue;
                // a cell top rounding onto the upper face spills into the next
                // column's first bin (see og_column_cells); keep the range in this column
                const int zc0 = s.u2c_min[f], zc1 = min(s.u2c_max[l], s.n_cells_z[col2] - 1);
                if (zc0 > zc1) continue;
                c2lo[ii] = head2 + zc0;
                c2hi[ii] = head2 + zc1;
            }
        }
        // The columns' candidates one after the other (column, image, cell: the list's order), a lane per
        // candidate, two chunks of 64 at a time.
        const int n0 = c2hi[0] - c2lo[0] + 1, n1 = c2hi[1] - c2lo[1] + 1, mine = n0 + n1 + c2hi[2] - c2lo[2] + 1;
        int       incl = mine;
        for (int off = 1; off < 64; off <<= 1) {
            const int v = __shfl_up(incl, off, 64);
            if (lane >= off) incl += v;
        }
        const int first = incl - mine, total = __builtin_amdgcn_readlane(incl, 63);
        T.at[lane]  = make_int4(first, c2lo[0] | imgxy << 24, c2lo[1], c2lo[2]);
        T.run[lane] = make_int3(n0, n1, __float_as_int(dd01));
        int owner = 0;  // of the last candidate of the chunk before
        for (int t0 = 0; t0 < total; t0 += 128) {
            int   c2[2], img[2];
            float zt[2], zb[2], dxy[2], sh[2];
            bool  in[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int t = t0 + 64 * j + lane, d = first - (t - lane);
                T.mark[lane] = 0;
                og_wave_lds();
                T.mark[mine > 0 && d >= 0 && d < 64 ? d : 64] = lane + 1;
                og_wave_lds();
                const int      v    = T.mark[lane];
                const uint64_t m    = __ballot(v != 0) & (~0ull >> (63 - lane));  // starts up to this candidate
                const int      from = __shfl(v, m ? 63 - __builtin_clzll(m) : lane, 64);
                const int      own  = m ? from - 1 : owner;
                owner               = __builtin_amdgcn_readlane(own, 63);
                const int4 at       = T.at[own];
                const int3 run      = T.run[own];
                const int  e = t - at.x, e1 = e - run.x, e2 = e1 - run.y;
                in[j]  = t < total;
                c2[j]  = e1 < 0 ? (at.y & 0xffffff) + e : e2 < 0 ? at.z + e1 : at.w + e2;
                c2[j]  = in[j] ? c2[j] : 0;
                img[j] = (at.y >> 24) | (e1 < 0 ? 16 : e2 < 0 ? 0 : 32);
                sh[j]  = (float)(e1 < 0 ? -1 : e2 < 0 ? 0 : 1) * s.L[2];
                dxy[j] = __int_as_float(run.z);
                zt[j]  = s.cell_zmax[c2[j]];
                zb[j]  = s.cell_zmin[c2[j]];
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const bool keep = in[j] && !(dxy[j] + og_zgap2(zt[j] + sh[j], zb[j] + sh[j], z1b, z1t) > s.cutoff_pair2) &&
                                  og_valid_pair(c1, c2[j]);
                const uint64_t m = __ballot(keep);
                if (keep) {
                    const int p   = pos + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                    const int rec = c2[j] | img[j] << 24;
                    if (MODE == 1) {
                        if (p < OG_ENUM_STAGE) s.cp_stage[(size_t)c1 * OG_ENUM_STAGE + p] = rec;
                    } else if (p < s.cap_cell_pairs) {
                        s.cp_c2[p] = rec;
                    }
                }
                pos += __builtin_popcountll(m);
            }
        }
        og_wave_lds();  // the next round overwrites the tables
    }
    if (MODE == 1 && lane == 0) *out_count = pos;
}

// One wave per cell.  SCAN: and the exclusive scan of the cells' pair counts
// over groups of 1,024 cells, by the last of a group's blocks (k_enum_scan's
// results).  That saves the scan's own launch; against it stand the blocks'
// wait for their stores and one counter per group (og_scan_with_count has both
// sides; 450,000 atoms 70 us per rebuild).
#define OG_SCAN_CELLS 1024
template <bool SCAN>
__global__ void __launch_bounds__(OG_THREADS) k_enum_count(const og_dev_sys *__restrict__ S,
                                                           const int2 *__restrict__ map) {
    __shared__ og_enum_lds lds[OG_THREADS / 64];
    const int2        bm = map[blockIdx.x];
    const og_dev_sys &s  = S[bm.x];
    if (og_rebuild_skip(s)) return;
    constexpr int PER = OG_THREADS / 64;  // cells per block
    const int     c0  = bm.y * PER, n = s.cnt->n_cells;
    const int     lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int     c1  = __builtin_amdgcn_readfirstlane(c0 + w);
    if (c0 >= n) return;
    if (c1 < n) {
        int count = 0;
        og_enum_cell<1>(s, lds[w], c1, 0, &count);
        if (lane == 0) {
            if (SCAN) __hip_atomic_store(&s.cp_count[c1], count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else s.cp_count[c1] = count;
        }
    }
    if (!SCAN) return;
    static_assert(OG_SCAN_CELLS % PER == 0 && OG_SCAN_CELLS == 4 * OG_THREADS, "whole blocks, four cells per thread");
    const int g = c0 / OG_SCAN_CELLS, g0 = g * OG_SCAN_CELLS, cells = min(OG_SCAN_CELLS, n - g0);
    if (!og_last_block(&s.cp_arrived[g], (cells + PER - 1) / PER)) return;
    int v[4], sum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = 4 * threadIdx.x + j;
        v[j] = c < cells ? __hip_atomic_load(&s.cp_count[g0 + c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) sum += v[j];
    __shared__ int wsum[PER];
    int            incl = sum;
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(incl, off, 64);
        if (lane >= off) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int at = incl - sum;
    for (int q = 0; q < w; q++) at += wsum[q];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = 4 * threadIdx.x + j;
        if (c < cells) s.cp_head[g0 + c] = at;
        at += v[j];
    }
    if (threadIdx.x == OG_THREADS - 1) s.cp_bsum[g] = at;
}

// Exclusive scan of the cells' pair counts, blocks of 1024 cells: each cell's
// prefix within its block to cp_head, the block's total to cp_bsum.  k_list
// adds the totals of the blocks before a cell's.
__global__ void __launch_bounds__(1024) k_enum_scan(const og_dev_sys *__restrict__ S,
                                                         const int2 *__restrict__ map) {
    const int2        bm = map ? map[blockIdx.x] : make_int2(0, (int)blockIdx.x);
    const og_dev_sys &s  = S[bm.x];
    if (og_rebuild_skip(s)) return;
    const int n = s.cnt->n_cells;
    if (bm.y * 1024 > n) return;
    const int k    = bm.y * 1024 + threadIdx.x;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __shared__ int wsum[16];
    const int      v    = k < n ? s.cp_count[k] : 0;
    int            incl = v;
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(incl, off, 64);
        if (lane >= off) incl += u;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0;
    for (int q = 0; q < w; q++) before += wsum[q];
    if (k < n) s.cp_head[k] = before + incl - v;
    if (threadIdx.x == 1023) s.cp_bsum[bm.y] = before + incl;
}

// ----------------------------------------------------------------- list --
// One wave per cell1: the cell's place in the list (its block prefix and the
// totals before), its records from the stage, and their masks.
//
// MiniCell::set_cell_pair_bitmask (MiniCell.cpp:1198-1237): bit a2*8+a1 set
// (= skip) for a dummy atom, the lower triangle of a self pair, or an nb15off
// partner (the partner list read up to its first -1).
// The exclusion bits are found from the atoms' side: the cell's partner
// lists are read once (lane = 8 * atom + partner) and each partner's grid
// slot becomes a (cell2, bit) entry in LDS; each lane then builds the masks
// of its share of the cell's pairs from the dummy flags, the self-pair
// triangle and the entries whose cell2 matches.  Same bits as testing every
// atom pair.
//
// A wave is a chain of memory round trips, so what does not depend on each
// other is read together: the counts, the first 64 staged records and the
// cell's atoms; then the records' atoms and the partner lists.  Offsets,
// records and masks took three kernels of such chains (450,000 atoms 110 us,
// now 84; 4,230 atoms 15 us and two launches more, now 9).
__global__ void __launch_bounds__(OG_THREADS, 8) k_list(const og_dev_sys *__restrict__ S, const int2 *__restrict__ map) {
    __shared__ union {
        og_enum_lds e;
        int         ex[OG_NAC * OG_MAX_NB15];  // (cell2 << 6) | bit
    } lds[OG_THREADS / 64];
    const int2        bm = map[blockIdx.x];
    const og_dev_sys &s  = S[bm.x];
    if (og_rebuild_skip(s)) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c1   = __builtin_amdgcn_readfirstlane(bm.y * (OG_THREADS / 64) + w);
    const int n    = s.cnt->n_cells;
    if (c1 >= n) return;
    int       *ex  = lds[w].ex;
    const int *src = s.cp_stage + (size_t)c1 * OG_ENUM_STAGE;
    const int  cnt = __builtin_amdgcn_readfirstlane(s.cp_count[c1]);
    int        rec = src[lane];  // the stage of a cell is longer than a wave
    static_assert(OG_ENUM_STAGE >= 64, "the first records are read before their count is known");
    const int  a1  = lane >> 3;
    const int  id1 = s.atomids[c1 * OG_NAC + a1];
    const int  idl = s.atomids[c1 * OG_NAC + (lane & 7)];
    long long  at  = 0;  // the list position of the cell's first record
    for (int q = lane; q < c1 / OG_SCAN_CELLS; q += 64) at += s.cp_bsum[q];
    for (int off = 32; off > 0; off >>= 1) at += __shfl_xor(at, off, 64);
    at += s.cp_head[c1];
    const long long end = at + cnt, cap = s.cap_cell_pairs;
    if (lane == 0) {
        s.cp_head[c1] = (int)min(at, cap);
        if (c1 == n - 1) {
            s.cp_head[n] = (int)min(end, cap);
            if (end > cap) atomicOr(&s.cnt->flags, OG_F_CP_OVERFLOW);
            s.cnt->n_cell_pairs = end > cap ? 0 : (int)end;
        }
    }
    const int  p0     = __builtin_amdgcn_readfirstlane((int)min(at, cap));
    const int  m1     = __builtin_amdgcn_readfirstlane((int)min(end, cap)) - p0;  // records that fit
    const bool staged = cnt <= OG_ENUM_STAGE;
    if (!staged) {  // did not fit the stage: enumerate again, writing in place
        og_enum_cell<2>(s, lds[w].e, c1, p0, nullptr);
        __threadfence_block();
        rec = lane < m1 ? s.cp_c2[p0 + lane] : 0;
    }
    const int4 *A4 = (const int4 *)s.atomids;
    int4        u  = make_int4(0, 0, 0, 0), v = u;
    if (lane < m1) u = A4[2 * (rec & 0xffffff)], v = A4[2 * (rec & 0xffffff) + 1];

    // exclusion entries: lane = 8 * a1 + (partner index within this round of 8)
    bool open = id1 >= 0;  // a1's list has not ended yet
    int  nex  = 0;
    for (int kb = 0; kb < OG_MAX_NB15; kb += 8) {
        const int      k    = kb + (lane & 7);
        const int      t    = open ? s.nb15off[(size_t)id1 * OG_MAX_NB15 + k] : -1;
        const uint64_t neg  = __ballot(open && t < 0);
        const unsigned term = (unsigned)(neg >> (8 * a1)) & 0xffu;  // -1 entries of a1 in this round
        const bool     keep = open && (lane & 7) < (term ? __builtin_ctz(term) : 8);
        open                = open && term == 0;
        const uint64_t kbal = __ballot(keep);
        if (keep) {
            const int g2   = s.rev[t];
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(kbal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)kbal, 0u));
            ex[nex + rank] = ((g2 >> 3) << 6) | ((g2 & 7) << 3) | a1;
        }
        nex += __builtin_popcountll(kbal);
        if (__ballot(open) == 0) break;
    }

    // dummy atoms of cell1: bit a1 of every row byte
    const unsigned dmy1 = (unsigned)__ballot(idl < 0) & 0xffu;
    const uint64_t cols = (uint64_t)dmy1 * 0x0101010101010101ull;
    // self pair: a1 >= a2, i.e. bits a2..7 of row byte a2
    uint64_t self = 0;
    for (int a2 = 0; a2 < OG_NAC; a2++) self |= (uint64_t)((0xffu << a2) & 0xffu) << (8 * a2);
    for (int base = 0; base < m1; base += 64) {
        const int k = base + lane;
        if (k < m1) {
            const int p  = p0 + k;
            const int c2 = rec & 0xffffff;
            uint64_t  m  = cols | (c2 == c1 ? self : 0ull);
            // dummy atoms of cell2: the whole row byte
            m |= (u.x < 0 ? 0xffull : 0ull) | (u.y < 0 ? 0xffull << 8 : 0ull) | (u.z < 0 ? 0xffull << 16 : 0ull) |
                 (u.w < 0 ? 0xffull << 24 : 0ull) | (v.x < 0 ? 0xffull << 32 : 0ull) |
                 (v.y < 0 ? 0xffull << 40 : 0ull) | (v.z < 0 ? 0xffull << 48 : 0ull) |
                 (v.w < 0 ? 0xffull << 56 : 0ull);
            for (int e = 0; e < nex; e++) {
                const int q = ex[e];
                if ((q >> 6) == c2) m |= 1ull << (q & 63);
            }
            if (staged) s.cp_c2[p] = rec;
            s.cp_mask[p] = m;
        }
        if (k + 64 < m1) {  // the next 64
            rec = staged ? src[k + 64] : s.cp_c2[p0 + k + 64];
            u   = A4[2 * (rec & 0xffffff)], v = A4[2 * (rec & 0xffffff) + 1];
        }
    }
}

// ------------------------------------------------------------- launchers --
void og_launch_grid_clear(const og_launch &cols) {
    hipLaunchKernelGGL(k_grid_clear, dim3(cols.n_blocks), dim3(OG_THREADS), 0, cols.stream, cols.sys, cols.map);
}
void og_launch_grid_bin(const og_launch &a, bool point) {
    hipLaunchKernelGGL(k_grid_bin, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, a.map, (int)point);
}
void og_launch_grid_scatter(const og_launch &a) {
    hipLaunchKernelGGL(k_grid_scatter, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, a.map);
}
void og_launch_grid_sort(const og_launch &a) {
    hipLaunchKernelGGL(k_grid_sort, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, a.map);
}
void og_launch_cells_from_grid(const og_launch &a) {
    hipLaunchKernelGGL(k_cells_from_grid, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, a.map);
}
void og_launch_enum_count(const og_launch &cellw, const og_launch &blocks, bool scan) {
    const dim3 nb(cellw.n_blocks), nt(OG_THREADS);
    if (scan) {
        hipLaunchKernelGGL(k_enum_count<true>, nb, nt, 0, cellw.stream, cellw.sys, cellw.map);
        return;
    }
    hipLaunchKernelGGL(k_enum_count<false>, nb, nt, 0, cellw.stream, cellw.sys, cellw.map);
    hipLaunchKernelGGL(k_enum_scan, dim3(blocks.n_blocks), dim3(1024), 0, blocks.stream, blocks.sys, blocks.map);
}
void og_launch_list(const og_launch &a) {
    hipLaunchKernelGGL(k_list, dim3(a.n_blocks), dim3(OG_THREADS), 0, a.stream, a.sys, a.map);
}
