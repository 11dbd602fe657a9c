// kst_output.hpp -- device side of the output diagnostics.
//
// CalculateVolume (src/Output.f90:617-735) sums over the active tiles' cells
// the flow volume (w - b0 - bt) gam^2, the mass rho Hn gam, the bed change bt
// and the solids Hnpsi gam (Hn and rho as ComputeDesingularisedVariables,
// src/HydraulicRHS.f90:762-878, derives them from the stored state).  The
// reference Kahan-sums them sequentially in active-list order.  Here each sum
// is a compensated parallel sum, Sum2 of Ogita, Rump and Oishi ("Accurate
// sum and dot product", SIAM J. Sci. Comput. 26, 2005): every addition is
// an error-free TwoSum (Knuth) whose rounding error is accumulated beside
// the running sum, partial (sum, error) pairs merge the same way, and the
// result is sum + error.  Its error is at most u|S| + gamma_{n-1}^2 sum|x_i|,
// so for these sums both it and the reference's Kahan sum lie within an ulp
// or two of the exact sum; the order of a launch is fixed by the active set,
// so the result is deterministic.
//
// The pass reads five FP64 words per active cell (w, Hnpsi, b0, bt, gam):
// an HBM-bound stream, one tile per workgroup iteration, coalesced along the
// tile's rows.
#pragma once

namespace kst {

constexpr int VOL_NT = 256;            // threads of a volume workgroup
constexpr int VOL_BLOCKS_MAX = 2048;   // partials of the first pass (8 XCDs x 256)
constexpr int VOL_Q = 4;               // flow volume, mass, bed, solids (in this order)

struct Sum2 {
    double s = 0.0, e = 0.0;
    __device__ __forceinline__ void add(double x) {
        const double t = s + x;
        const double z = t - s;
        e = e + ((s - (t - z)) + (x - z));
        s = t;
    }
    __device__ __forceinline__ void merge(double s2, double e2) {
        add(s2);
        e = e + e2;
    }
};

// Both halves of a double through a lane exchange of 32-bit words.
template <class F>
__device__ __forceinline__ double each_half(double x, F f) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = f((unsigned)b), hi = f((unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Lane l of each row of 16 takes lane l + N's value (0 beyond the row).
template <int N>
__device__ __forceinline__ double from_above(double x) {
    return each_half(x, [](unsigned v) {
        return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x100 + N, 0xf, 0xf, true);
    });
}

// Where bit N (16 or 32) of the lane index is 0, a and b become a of this lane
// and of the lane N above; where it is 1, b of the lane N below and of this one.
template <int N>
__device__ __forceinline__ void swap_halves(double& a, double& b) {
    unsigned long long x = (unsigned long long)__double_as_longlong(a), y = (unsigned long long)__double_as_longlong(b);
    unsigned w[2][2];
    for (int k = 0; k < 2; ++k) {
        const unsigned u = (unsigned)(x >> (32 * k)), v = (unsigned)(y >> (32 * k));
        const auto r = N == 32 ? __builtin_amdgcn_permlane32_swap(u, v, false, false)
                               : __builtin_amdgcn_permlane16_swap(u, v, false, false);
        w[0][k] = r[0];
        w[1][k] = r[1];
    }
    a = __longlong_as_double((long long)(((unsigned long long)w[0][1] << 32) | w[0][0]));
    b = __longlong_as_double((long long)(((unsigned long long)w[1][1] << 32) | w[1][0]));
}

template <int N>
__device__ __forceinline__ Sum2 split_merge(Sum2 a, Sum2 b) {
    swap_halves<N>(a.s, b.s);
    swap_halves<N>(a.e, b.e);
    a.merge(b.s, b.e);      // the lower lane's pair first, on either side
    return a;
}
template <int N>
__device__ __forceinline__ void row_merge(Sum2& a) {
    const double s2 = from_above<N>(a.s), e2 = from_above<N>(a.e);
    a.merge(s2, e2);
}

// Merges the VOL_Q pairs of a workgroup; thread q < VOL_Q returns pair q.
// Within a wave the tree of lane pairs 32, 16, 8, 4, 2, 1 apart: the first two
// steps also share the four sums out over the wave's rows of 16 lanes, so that
// a wave does 7 merges, not 24 (the reduction was half of the kernel's
// instructions: a workgroup has one tile, 4 cells a thread).
__device__ __forceinline__ Sum2 vol_block_reduce(const Sum2 (&a)[VOL_Q], double* sh) {
    static_assert(VOL_Q == 4, "one row of 16 lanes per sum");
    const Sum2 lo = split_merge<32>(a[0], a[2]), hi = split_merge<32>(a[1], a[3]);
    Sum2 m = split_merge<16>(lo, hi);
    row_merge<8>(m);
    row_merge<4>(m);
    row_merge<2>(m);
    row_merge<1>(m);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if ((lane & 15) == 0) {
        sh[(wv * VOL_Q + lane / 16) * 2] = m.s;
        sh[(wv * VOL_Q + lane / 16) * 2 + 1] = m.e;
    }
    __syncthreads();
    Sum2 r;
    if (threadIdx.x < VOL_Q) {
        r.s = sh[threadIdx.x * 2];
        r.e = sh[threadIdx.x * 2 + 1];
        for (int w = 1; w < VOL_NT / 64; ++w)
            r.merge(sh[(w * VOL_Q + threadIdx.x) * 2], sh[(w * VOL_Q + threadIdx.x) * 2 + 1]);
    }
    return r;
}

// The partials of an active set of n tiles.
__host__ __device__ __forceinline__ int volume_partials(int n) { return n < 1 ? 1 : (n < VOL_BLOCKS_MAX ? n : VOL_BLOCKS_MAX); }

// First pass: of G = volume_partials(active tiles) workgroups, b takes
// active-list entries b, b + G, ... and writes its VOL_Q (sum, error) pairs to
// part[b].  The grid covers every tile of the domain (up to the partials'
// capacity), so that the host need not read the active set first; the
// workgroups beyond G end.
__global__ __launch_bounds__(VOL_NT) void volume_kernel(const Dev* dA, const Params* pA, double* part) {
    const auto& d = const_arg(dA);
    const auto& p = const_arg(pA);
    __shared__ double sh[VOL_NT / 64 * VOL_Q * 2];
    const auto* c = ctrl_view(d);
    const int na = c->n_active, G = volume_partials(na);
    if ((int)blockIdx.x >= G) return;
    const bool flat = c->flat != 0;      // bt is 0 everywhere
    // mixed precision: u^n is in S0 or S0b by Ctrl::cur
    const double* Sn = (d.mixed && c->cur) ? d.S0b : d.S0;
    const long long FS = d.FS;
    const int NC = p.NC;
    const double eps2 = p.hthr * p.hthr;
    constexpr int U = 4;                 // cells a thread loads at once
    Sum2 a[VOL_Q];
    for (int it = blockIdx.x; it < na; it += G) {
        const size_t base = (size_t)d.active[it] * NC;
        for (int i0 = threadIdx.x; i0 < NC; i0 += U * VOL_NT) {
            double w[U], hp[U], b0[U], bt[U], gam[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const unsigned g = (unsigned)(base + min(i0 + k * VOL_NT, NC - 1));
                w[k] = ld(Sn, g);
                hp[k] = ld(Sn + 3 * FS, g);
                b0[k] = ld(d.b0c, g);
                bt[k] = flat ? 0.0 : ld(d.TA.btc, g);
                gam[k] = ld(d.TA.cgam, g);
            }
#pragma unroll
            for (int k = 0; k < U; ++k) {
                if (i0 + k * VOL_NT >= NC) break;
                // (w - b0 - bt) gam gam, evaluated left to right
                double dv = w[k] - b0[k];
                dv = dv - bt[k];
                dv = dv * gam[k];
                dv = dv * gam[k];
                double hn = compute_hn(w[k], b0[k], bt[k], gam[k]);
                if (hn < 0.0) hn = 0.0;
                const double hpc = hp[k] < 0.0 ? 0.0 : hp[k];
                const double psi = dmin(2.0 * hn * hpc / (hn * hn + dmax(hn * hn, eps2)), p.max_pack);
                const double rho = density(generic(p), psi);
                a[0].add(dv);
                a[1].add(rho * hn * gam[k]);
                a[2].add(bt[k]);
                a[3].add(hp[k] * gam[k]);
            }
        }
    }
    const Sum2 r = vol_block_reduce(a, sh);
    if (threadIdx.x < VOL_Q) {
        part[(size_t)blockIdx.x * VOL_Q * 2 + 2 * threadIdx.x] = r.s;
        part[(size_t)blockIdx.x * VOL_Q * 2 + 2 * threadIdx.x + 1] = r.e;
    }
}

// Second pass: one workgroup merges the partials (thread t takes t,
// t + VOL_NT, ...) and writes the VOL_Q pairs to out.
__global__ __launch_bounds__(VOL_NT) void volume_final_kernel(const Dev* dA, const double* part, double* out) {
    __shared__ double sh[VOL_NT / 64 * VOL_Q * 2];
    const int nb = volume_partials(ctrl_view(const_arg(dA))->n_active);
    Sum2 a[VOL_Q];
    for (int b = threadIdx.x; b < nb; b += VOL_NT)
        for (int q = 0; q < VOL_Q; ++q)
            a[q].merge(part[(size_t)b * VOL_Q * 2 + 2 * q], part[(size_t)b * VOL_Q * 2 + 2 * q + 1]);
    const Sum2 r = vol_block_reduce(a, sh);
    if (threadIdx.x < VOL_Q) {
        out[2 * threadIdx.x] = r.s;
        out[2 * threadIdx.x + 1] = r.e;
    }
}

// ---------------------------------------------------------------------------
// OutputSolutionData_txt (src/Output.f90:754-929): per active cell, in the
// order of the file's columns 6-19, flow depth Hn, flow speed, u, v, rho,
// psi, rhoHnu, rhoHnv, Hnpsi, w, b0, bt, db/dx, db/dy, as tileContainer holds
// them.  Hn, psi and rho are its desingularised variables
// (ComputeDesingularisedVariables, src/HydraulicRHS.f90:762-878, evaluated as
// the reference orders it), which the final implicit pass leaves consistent
// with w and Hnpsi; u and v are the ones the step's last RHS derived (Dev::UVo),
// since that pass changes the momentum after them.  The speed is
// sqrt(FlowSquaredSpeedSlopeAligned) of those where Hn exceeds the height
// threshold, else 0 (src/Output.f90:868-873).  out[list position][column][cell].
// ---------------------------------------------------------------------------

constexpr int OUT_COLS = 14;

// tileContainer's velocities after kst_set_state: desingularised from the
// state (the reference's set-up ends with ComputeDesingularisedVariables on
// the active tiles).
__global__ __launch_bounds__(VOL_NT) void uv_init_kernel(const Dev* dA, const Params* pA) {
    const auto& d = const_arg(dA);
    const auto& p = const_arg(pA);
    const auto* c = ctrl_view(d);
    const int na = c->n_active;
    const double* Sn = (d.mixed && c->cur) ? d.S0b : d.S0;
    const long long FS = d.FS;
    const int NC = p.NC;
    const double eps = p.hthr;
    for (int it = blockIdx.x; it < na; it += gridDim.x) {
        const long long base = (long long)d.active[it] * NC;
        for (int i = threadIdx.x; i < NC; i += VOL_NT) {
            const long long g = base + i;
            const double w = Sn[g], ru = Sn[FS + g], rv = Sn[2 * FS + g], hp = Sn[3 * FS + g];
            double hn = compute_hn(w, d.b0c[g], d.TA.btc[g], d.TA.cgam[g]);
            if (hn < 0.0) hn = 0.0;
            const double hpc = hp < 0.0 ? 0.0 : hp;
            const double psi = dmin(2.0 * hn * hpc / (hn * hn + dmax(hn * hn, eps * eps)), p.max_pack);
            const double rho = density(generic(p), psi);
            d.UVo[g] = 2.0 * hn * ru / (hn * hn + dmax(hn * hn, eps * eps)) / rho;
            // a 1D grid never derives v (src/HydraulicRHS.f90:870-874)
            d.UVo[FS + g] = p.oned ? 0.0 : 2.0 * hn * rv / (hn * hn + dmax(hn * hn, eps * eps)) / rho;
        }
    }
}

__global__ __launch_bounds__(VOL_NT) void output_kernel(const Dev* dA, const Params* pA, double* out) {
    const auto& d = const_arg(dA);
    const auto& p = const_arg(pA);
    const auto* c = ctrl_view(d);
    const int na = c->n_active;
    const double* Sn = (d.mixed && c->cur) ? d.S0b : d.S0;
    const long long FS = d.FS;
    const int NC = p.NC;
    const double eps = p.hthr;
    for (int it = blockIdx.x; it < na; it += gridDim.x) {
        const long long base = (long long)d.active[it] * NC;
        double* o = out + (size_t)it * OUT_COLS * NC;
        for (int i = threadIdx.x; i < NC; i += VOL_NT) {
            const long long g = base + i;
            const double w = Sn[g], ru = Sn[FS + g], rv = Sn[2 * FS + g], hp = Sn[3 * FS + g];
            const double b0 = d.b0c[g], bt = d.TA.btc[g], bx = d.TA.cbx[g], by = d.TA.cby[g];
            const double gam = d.TA.cgam[g];
            double hn = compute_hn(w, b0, bt, gam);
            if (hn < 0.0) hn = 0.0;
            const double hpc = hp < 0.0 ? 0.0 : hp;
            const double psi = dmin(2.0 * hn * hpc / (hn * hn + dmax(hn * hn, eps * eps)), p.max_pack);
            const double rho = density(generic(p), psi);
            const double uu = d.UVo[g], vv = d.UVo[FS + g];
            const double spd = hn > p.hthr ? sqrt(speed2(p.geometric, uu, vv, bx, by)) : 0.0;
            const double col[OUT_COLS] = {hn, spd, uu, vv, rho, psi, ru, rv, hp, w, b0, bt, bx, by};
#pragma unroll
            for (int q = 0; q < OUT_COLS; ++q) o[(size_t)q * NC + i] = col[q];
        }
    }
}

}  // namespace kst
