// kst_io.hpp -- the boundary's row-major arrays <-> the tile-major layout, on
// the device.  The host arrays of the C-ABI hold a grid row by row; the step
// keeps each tile's cells (vertices) together.  Arrays cross the link as they
// are, once, through the device's staging (Stage), and these kernels rearrange
// them and fill every buffer that starts from the state, a chunk of the
// row-major arrays -- elements [g0, g0 + n), in the staging from 0 on -- at a
// time.  They are bound by HBM (a 2048 x 2048 set-up writes 1.1 GB in 0.3 ms);
// rearranged on one host thread, with each buffer filled by a copy of its own,
// the same set-up took 134 ms and reading the state 141 ms.  Included by
// kst_step.hip.
#pragma once

namespace kst {

constexpr int IO_NT = 256;

// Tile-major place of the row-major cell g, and its tile.
__device__ __forceinline__ size_t tile_major(const Params& p, size_t g, int& t) {
    const int NX = p.ntx * p.nx;
    const int J = (int)(g / NX), I = (int)(g % NX);
    t = I / p.nx + (J / p.ny) * p.ntx;
    return (size_t)t * p.NC + (J % p.ny) * p.nx + I % p.nx;
}

// Vertices: every tile's own copy of the global values; with `active` only
// the active tiles take them, the others 0 (ghost tiles keep bt = 0, as
// AllocateTopographicData leaves them).  in = nullptr: 0 everywhere.  Tiles
// t0, t0 + 1, ... by the block; vertices of other chunks stay as they are.
struct VertexSets {
    double* v[4];
    int n;
};
__global__ __launch_bounds__(IO_NT) void scatter_vertices_kernel(Params p, const double* in, const uint8_t* active,
                                                                 VertexSets out, int t0, size_t g0, size_t n) {
    const int t = t0 + blockIdx.x, NV1 = p.nx + 1, NV = NV1 * (p.ny + 1);
    const int ti = t % p.ntx, tj = t / p.ntx;
    const size_t GX = (size_t)p.ntx * p.nx + 1;
    const bool take = in && (!active || active[t] == KST_TILE_ACTIVE);
    for (int q = threadIdx.x; q < NV; q += IO_NT) {
        const int i = q % NV1, j = q / NV1;
        const size_t g = (size_t)(tj * p.ny + j) * GX + ti * p.nx + i - g0;   // wraps below g0
        if (g >= n) continue;
        const double v = take ? in[g] : 0.0;
        for (int k = 0; k < out.n; ++k) out.v[k][(size_t)t * NV + q] = v;
    }
}

// The state of a fresh run in every buffer that holds one.  in: w, rhoHnu,
// rhoHnv, Hnpsi (and the initial maximum of Hn), n apart.  Active tiles take
// it; ghost tiles hold the data of UpdateGhostTileBCs (new_tile_cell), the
// others dry data.  The maxima start afresh.
__global__ __launch_bounds__(IO_NT) void scatter_state_kernel(Dev d, Params p, const double* in, int have_hn,
                                                              size_t g0, size_t n) {
    const size_t FS = (size_t)d.FS;
    for (size_t i = (size_t)blockIdx.x * IO_NT + threadIdx.x; i < n; i += (size_t)gridDim.x * IO_NT) {
        int t;
        const size_t gi = tile_major(p, g0 + i, t);
        const uint8_t st = d.tstate[t];
        CellData v;
        if (st == KST_TILE_ACTIVE) v = {in[i], in[n + i], in[2 * n + i], in[3 * n + i]};
        else v = new_tile_cell(d, p, t, gi, st != KST_TILE_GHOST);
        const double f[4] = {v.w, v.ru, v.rv, v.hp};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const size_t k = q * FS + gi;
            d.S0[k] = f[q];
            if (d.mixed) {
                d.S0b[k] = f[q];
                ((float*)d.S2)[k] = 0.f;
                ((float*)d.S3)[k] = 0.f;
            } else {
                d.S2[k] = f[q];
                d.S3[k] = f[q];
            }
            if (d.morpho) d.SH[k] = f[q];
        }
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            if (d.mixed) ((float*)d.R)[q * FS + gi] = 0.f;
            else d.R[q * FS + gi] = 0.0;
            if (d.morpho) d.R2[q * FS + gi] = 0.0;
        }
        if (d.morpho) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                d.SM[q][gi] = v.w;
                d.SM[q][FS + gi] = v.hp;
            }
            d.UV[gi] = 0.0;
            d.UV[FS + gi] = 0.0;
        }
        d.gsx[gi] = 0.0;
        d.gsy[gi] = 0.0;
        d.UVo[gi] = 0.0;
        d.UVo[FS + gi] = 0.0;
#pragma unroll
        for (int q = 1; q < 10; ++q) d.maxima[q * FS + gi] = 0.0;
        d.maxima[gi] = have_hn ? in[4 * n + i] : 0.0;
        d.maxima[10 * FS + gi] = -1.0;
    }
}

// One cell array in (mask: only where it is not 0) or out (ts: 0 outside
// allocated tiles).
__global__ __launch_bounds__(IO_NT) void scatter_cells_kernel(Params p, const double* in, const uint8_t* mask,
                                                              double* out, size_t g0, size_t n) {
    for (size_t i = (size_t)blockIdx.x * IO_NT + threadIdx.x; i < n; i += (size_t)gridDim.x * IO_NT) {
        int t;
        const size_t k = tile_major(p, g0 + i, t);
        if (!mask || mask[i]) out[k] = in[i];
    }
}
__global__ __launch_bounds__(IO_NT) void gather_cells_kernel(Params p, const double* in, double* out, size_t g0,
                                                             size_t n) {
    for (size_t i = (size_t)blockIdx.x * IO_NT + threadIdx.x; i < n; i += (size_t)gridDim.x * IO_NT) {
        int t;
        out[i] = in[tile_major(p, g0 + i, t)];
    }
}

// What kst_get_state returns, six arrays n apart: w, rhoHnu, rhoHnv, Hnpsi (0
// outside allocated tiles) and Hn ((w - b0 - bt) gamma where positive in active tiles;
// a ghost's is the one it was given: zero, or the Dirichlet boundary depth on
// the domain edge), then the vertex bt -- vertex (I, J) from the copy of the
// tile holding cell (min(I, NX-1), min(J, NY-1)) -- and the time behind them.
// (There are more vertices than cells: the chunk is one of vertices.)
__global__ __launch_bounds__(IO_NT) void gather_state_kernel(Dev d, Params p, double* out, size_t g0, size_t n) {
    const size_t FS = (size_t)d.FS;
    const double* S = d.mixed && d.ctrl->cur ? d.S0b : d.S0;
    const int NX = p.ntx * p.nx, NY = p.nty * p.ny, NV1 = p.nx + 1;
    const size_t NV = (size_t)NV1 * (p.ny + 1);
    for (size_t i = (size_t)blockIdx.x * IO_NT + threadIdx.x; i < n; i += (size_t)gridDim.x * IO_NT) {
        const size_t g = g0 + i;
        if (g < FS) {
            int t;
            const size_t k = tile_major(p, g, t);
            const uint8_t st = d.tstate[t];
            const bool held = st != KST_TILE_OFF;
            const double w = S[k];
            out[i] = held ? w : 0.0;
#pragma unroll
            for (int q = 1; q < 4; ++q) out[q * n + i] = held ? S[q * FS + k] : 0.0;
            double h = 0.0;
            if (st == KST_TILE_GHOST) {
                if (dirichlet_ghost(p, t)) h = p.bc_hn;
            } else if (st == KST_TILE_ACTIVE) {
                h = compute_hn(w, d.b0c[k], d.TA.btc[k], d.TA.cgam[k]);
                if (h < 0.0) h = 0.0;
            }
            out[4 * n + i] = h;
        }
        const int J = (int)(g / (NX + 1)), I = (int)(g % (NX + 1));
        const int gi = min(I, NX - 1) / p.nx, gj = min(J, NY - 1) / p.ny, t = gi + gj * p.ntx;
        out[5 * n + i] =
            d.tstate[t] == KST_TILE_OFF ? 0.0 : d.TA.vbt[(size_t)t * NV + (J - gj * p.ny) * NV1 + I - gi * p.nx];
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) out[6 * n] = d.ctrl->t;
}

}  // namespace kst
