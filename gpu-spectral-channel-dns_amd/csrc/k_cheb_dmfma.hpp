// k_cheb_dmfma.hpp -- the padded p2s of the FP64 form as dense FP64 products on the matrix
// cores (v_mfma_f64_16x16x4_f64), with the Chebyshev derivative, the nonlinear combination
// and the unpadded s2p folded into the tables.
//
// Reference counterparts: the padded p2s of the three Lamb components (cheby_p2s,
// source/transform.cu:538-658), rhsNonlinear (source/nonlinear.cu:146-242) and the unpadded
// s2p of N_v, N_eta (source/rhs.cpp:96-97); the (0,0) pencil keeps L_x, L_y at the nz points
// (source/rhs.cpp:229-236).
//
// With P the padded p2s (pz = 2N + 1 samples -> nz coefficients), D the Chebyshev
// derivative and S the values at the nz collocation points, M0 = S P and M1 = S D P map the
// samples of a component straight to the nz points.  rhsNonlinear is linear in the three
// components, so per pencil (alpha, beta, k^2 = alpha^2 + beta^2)
//   N_v   = M0 h1 + M1 h2,   h1 = k^2 f_z,   h2 = i alpha f_x + i beta f_y
//   N_eta = M0 h3,           h3 = i alpha f_y - i beta f_x
// (pencil (0,0): h1 = f_x, h2 = 0, h3 = f_y).  Reflection parity folds every product: with
// G+_q = f_q + f_{2N-q} (q < N; G+_N = f_N) and G-_q = f_q - f_{2N-q}, row p <= N/2 of a
// product is S_p + A_p and row N - p is S_p - A_p, where S = Q0s G+ (or Q1s G- for M1) over
// the "sym" rows p <= N/2 and A = Q0a G- (Q1a G+) over the "anti" rows p < N/2.  The tables
// are computed once per length on the host in long double and rounded to FP64.
//
// MFMA operand layouts of v_mfma_f64_16x16x4_f64 (checked on the GPU): lane l holds
// A[l % 16][l / 16], B[l / 16][l % 16], and D[l / 16 + 4 r][l % 16] for r < 4.  Tables are
// stored as fragments (row tile, k-step) of 64 doubles in this lane order.
#pragma once
#include "k_transform.hpp"

namespace cheb_dmfma {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int kPencils = 16;  // pencils per item: columns 0..15 real parts, 16..31 imaginary parts
constexpr int kCols = 2 * kPencils;
// samples q per chunk of the product's inner dimension, at most: 16 leave room for a fourth and
// fifth block per CU, 32 halve a block's serial chunks.  k_p2s_dmfma with 32 / 16 (us): 256x97x256
// (2064 blocks) 185 / 156, 128x129x128 (1040) 73 / 65, 128x65x128 (520) 29.2 / 27.8, 64x193x64 (264)
// 71 / 57; 64x65x64 (132) 15.1 / 16.1, 32x129x32 (68) 21.2 / 23.3, 32x33x32 (34) 11.9 / 12.3: 16
// where the blocks outnumber the compute units.
constexpr int kChunk = 32, kChunkMany = 16;

constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }

template <int FN, int CH = kChunk>
struct DShape {
    static constexpr int N = FN / 2, nz = N + 1, pz = FN + 1;
    static constexpr int RS = N / 2 + 1, RA = N / 2;  // sym rows p <= N/2, anti rows p < N/2
    // a centre row N/2 that starts a row tile of its own is a dot product on the vector units
    static constexpr bool CENTRE = (N / 2) % 16 == 0;
    static constexpr int RTS = ceil_div(RS, 16), RTA = ceil_div(RA, 16);
    static constexpr int RTM = CENTRE ? RTS - 1 : RTS;  // sym row tiles on the matrix cores
    static constexpr int NPAIR = RTM > RTA ? RTM : RTA;  // row tiles of each kind
    static_assert(RTM == RTA, "the sym and anti row tiles pair up");
    // a block takes TPB sym and TPB anti row tiles of an item (H blocks per item): one wave
    // per tile, each wave over both column tiles (real and imaginary parts)
    static constexpr int TPB = NPAIR > 2 && NPAIR % 2 == 0 ? NPAIR / 2 : NPAIR;
    static constexpr int H = NPAIR / TPB;
    static constexpr int NT = 128 * TPB;
    static constexpr int KP = ceil_div(N + 1, 4), KM = ceil_div(N, 4);  // k-steps of the tables over G+, G-
    // The chunks cover the samples q < N (N/4 k-steps of both G+ and G-); the centre sample
    // q = N (G+ only) is a rank-one update on the vector units.  Samples per chunk: the largest
    // multiple of 4 dividing N, at most CH.
    static constexpr int chunk_of(int n) {
        for (int c = CH; c >= 4; c -= 4)
            if (n % c == 0) return c;
        return 0;
    }
    static constexpr int CHK = chunk_of(N);
    static_assert(CHK > 0, "N divisible by 4");
    static constexpr int KPC = CHK / 4;  // k-steps per chunk
    static constexpr int NCH = N / CHK;
    static constexpr int UPT = ceil_div(CHK * kPencils, NT);  // (q, pencil) units per thread and chunk
    // fragment offsets (in fragments of 64 doubles): Q0s [RTS][KP], Q0a [RTA][KM], Q1s [RTS][KM],
    // Q1a [RTA][KP]; then the centre rows Q0s[N/2][0..N] and Q1s[N/2][0..N-1], and the
    // columns of the centre sample Q0s[0..N/2][N] and Q1a[0..N/2-1][N], as plain doubles
    static constexpr long F0S = 0, F0A = F0S + (long)RTS * KP, F1S = F0A + (long)RTA * KM,
                          F1A = F1S + (long)RTS * KM, FEND = F1A + (long)RTA * KP;
    static constexpr long CENTRE_OFF = FEND * 64;
    static constexpr long COLN_OFF = CENTRE_OFF + (N + 1) + N;
    static constexpr long table_doubles = COLN_OFF + RS + RA;
    // LDS: the operand buffer [set h3, h2, h1][G+, G-][CHK][kCols] doubles, reused after the
    // last chunk to stage the block's output rows [pencil][SR][re, im] of N_v, then of N_eta:
    // rows p of its tiles, their mirrors N - p and the centre row
    static constexpr int BUF = 3 * 2 * CHK * kCols;
    static constexpr int SR = 32 * TPB + 1;
    static constexpr size_t lds_bytes() {
        const size_t ops = (size_t)BUF * sizeof(double);
        const size_t out = (size_t)kPencils * SR * 2 * sizeof(double);
        return ops > out ? ops : out;
    }
    // blocks for nitems items: groups of 8 items, the H blocks of an item 8 ids apart (the
    // same XCD, dispatched together, so the item's samples are read from HBM once)
    static int blocks(int nitems) { return (nitems + 7) / 8 * 8 * H; }
};

}  // namespace cheb_dmfma

// -------------------------------------------------------------------------------------
// Padded p2s + derivative + rhsNonlinear + unpadded s2p of the FP64 form: Z1[3][kx][q][ky]
// (the three Lamb components after the span transform, q = 0..2N) -> N_v, N_eta at the nz
// points, FP64, in the slot's current history buffers.  An item is (member, kx, 16
// consecutive ky); block (item, h) computes the rows of sym and anti row tiles
// h TPB .. h TPB + TPB - 1 (and their mirrors N - p), in NCH chunks of CHK samples q < N
// (with their mirrors 2N - q).  Per chunk: thread units (q, pencil) fold the six samples of
// x, y, z (loaded one chunk ahead) into G+ and G-, combine them into h3, h2, h1 and write them
// as B operands to LDS; the waves load their table fragments (from L2); after a barrier each
// wave runs the chunk's k-steps for its tile over both column tiles -- Q0 fragments serve h3
// and h1, Q1 fragments h2 -- while the next chunk's samples are in flight.  The centre
// sample q = N enters afterwards as a rank-one update of the accumulators on the vector
// units.  Several blocks share a compute unit, so one block's products overlap another's
// loads.  At the end the
// sym waves write S to rows p and N - p of an LDS stage, the anti waves add A to row p and
// subtract it from row N - p, and the rows leave as contiguous runs of the pencils.  A
// centre row N/2 of its own runs on the vector units from the same LDS operands.
// -------------------------------------------------------------------------------------
template <int FN, int CH>
__global__ __launch_bounds__((cheb_dmfma::DShape<FN, CH>::NT), 3) void k_p2s_dmfma(
    const double2* __restrict__ Z1, long zstride, long sY, double2* __restrict__ NL, long sNL, Dims d,
    const double* __restrict__ tab, Members mb, int nitems, int nyb) {
    using namespace cheb_dmfma;
    using Sh = DShape<FN, CH>;
    constexpr int N = Sh::N, nz = Sh::nz, NT = Sh::NT, UPT = Sh::UPT, CHK = Sh::CHK, TPB = Sh::TPB, SR = Sh::SR;
    RPCF_LDS(double);
    __shared__ double cpart[2 * TPB][2][32];  // centre row: per wave, [N_eta, N_v][column]
    // centre row weights Q0s[N/2][0..N], Q1s[N/2][0..N-1]
    __shared__ double ctr[Sh::CENTRE ? 2 * N + 1 : 1];
    // block -> (item, h): groups of 8 items, the H blocks of an item 8 ids apart
    const int grp = blockIdx.x / (8 * Sh::H), rem8 = blockIdx.x % (8 * Sh::H);
    const int item = grp * 8 + rem8 % 8, h = rem8 / 8;
    if (item >= nitems) return;
    const bool centre = Sh::CENTRE && h == Sh::H - 1;  // this block also computes row N/2
    // waves 0 .. TPB-1: sym row tiles h TPB + wave; waves TPB .. 2 TPB-1: the anti row tiles
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: branches on it are scalar
    const bool anti = wave >= TPB;
    const int rt = h * TPB + (anti ? wave - TPB : wave);
    const int kq = lane >> 4, lc = lane & 15;
    const v4d zero4 = {0.0, 0.0, 0.0, 0.0};

    int slot, kx, ky0, nb;
    {
        const int per = d.hnx * nyb;
        const int m = item / per, r = item - m * per;
        slot = mb.ids[m];
        kx = r / nyb;
        ky0 = (r - kx * nyb) * kPencils;
        nb = min(kPencils, d.ny - ky0);
    }
    const double2* in = Z1 + slot * sY + (long)kx * Sh::pz * d.ny + ky0;
    // registers: the samples q and 2N - q of x, y, z for this thread's units of one chunk
    double2 sa[UPT][3], sb[UPT][3];
    auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int i = tid + u * NT, q = c * CHK + i / kPencils, b = i % kPencils;
            const bool ok = i < CHK * kPencils && b < nb;
            const long oa = ok ? (long)q * d.ny + b : 0, ob = ok ? (long)(FN - q) * d.ny + b : 0;
#pragma unroll
            for (int g = 0; g < 3; g++) {
                sa[u][g] = in[g * zstride + oa];
                sb[u][g] = in[g * zstride + ob];
            }
        }
    };
    const double aphi = mb.mp[slot].aphi, beta = mb.mp[slot].beta;
    // h3 = i alpha y - i beta x, h2 = i alpha x + i beta y, h1 = k^2 z of pencil ky0 + b
    // (pencil (0,0): y, 0, x)
    auto combine = [&](double2 x, double2 y, double2 z, int b, double2* h3, double2* h2, double2* h1) {
        const int ky = ky0 + b;
        const double ia = (double)kx / aphi;
        const double ib = ky >= d.ny / 2 + 1 ? (double)(ky - d.ny) / beta : (double)ky / beta;
        const double k2 = ia * ia + ib * ib;
        const bool mean = kx == 0 && ky == 0;
        // i a y - i b x = (-a y.im + b x.im, a y.re - b x.re); i a x + i b y likewise
        *h3 = mean ? y : make_double2(-ia * y.y + ib * x.y, ia * y.x - ib * x.x);
        *h2 = mean ? make_double2(0.0, 0.0) : make_double2(-ia * x.y - ib * y.y, ia * x.x + ib * y.x);
        *h1 = mean ? x : make_double2(k2 * z.x, k2 * z.y);
    };
    // the centre sample q = N of every pencil, combined: hN[set h3, h2, h1][column]
    __shared__ double hN[3][kCols];
    if (tid < kPencils) {
        double2 h3 = make_double2(0.0, 0.0), h2 = h3, h1 = h3;
        if (tid < nb) {
            const long o = (long)N * d.ny + tid;
            combine(in[o], in[zstride + o], in[2 * zstride + o], tid, &h3, &h2, &h1);
        }
        hN[0][tid] = h3.x, hN[0][kPencils + tid] = h3.y;
        hN[1][tid] = h2.x, hN[1][kPencils + tid] = h2.y;
        hN[2][tid] = h1.x, hN[2][kPencils + tid] = h1.y;
    }
    // fold, combine and write the B operands of chunk c
    auto stage = [&](int c) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int i = tid + u * NT;
            if (i >= CHK * kPencils) continue;
            const int qq = i / kPencils, b = i % kPencils;
            const bool ok = b < nb;
            double2 gp[3], gm[3];
#pragma unroll
            for (int g = 0; g < 3; g++) {
                const double2 a = sa[u][g], m = sb[u][g];
                gp[g] = ok ? make_double2(a.x + m.x, a.y + m.y) : make_double2(0.0, 0.0);
                gm[g] = ok ? make_double2(a.x - m.x, a.y - m.y) : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int pm = 0; pm < 2; pm++) {
                double2 h3, h2, h1;
                combine(pm ? gm[0] : gp[0], pm ? gm[1] : gp[1], pm ? gm[2] : gp[2], b, &h3, &h2, &h1);
                double* o = lds + (pm * CHK + qq) * kCols + b;
                o[0] = h3.x;
                o[kPencils] = h3.y;
                o[2 * CHK * kCols] = h2.x;
                o[2 * CHK * kCols + kPencils] = h2.y;
                o[4 * CHK * kCols] = h1.x;
                o[4 * CHK * kCols + kPencils] = h1.y;
            }
        }
    };
    // this wave's tables: sym: Q0 = Q0s over G+, Q1 = Q1s over G-; anti: Q0 = Q0a over G-,
    // Q1 = Q1a over G+
    const double* tq0 = tab + (anti ? Sh::F0A + (long)rt * Sh::KM : Sh::F0S + (long)rt * Sh::KP) * 64 + lane;
    const double* tq1 = tab + (anti ? Sh::F1A + (long)rt * Sh::KP : Sh::F1S + (long)rt * Sh::KM) * 64 + lane;
    const int pm0 = anti ? 1 : 0;  // side of h3, h1 (Q0) for this wave; h2 (Q1) takes the other
    // B operand of lane (kq, lc) at local k-step sl of set s, side pm, column tile ct
    auto bop = [&](int s, int pm, int sl, int ct) {
        return lds[((s * 2 + pm) * CHK + 4 * sl + kq) * kCols + ct * kPencils + lc];
    };
    if (centre) {
        for (int i = tid; i < 2 * N + 1; i += NT) ctr[i] = tab[Sh::CENTRE_OFF + i];
    }
    // accumulators [column tile] of N_eta and N_v over this wave's rows (S or A)
    v4d accE[2] = {zero4, zero4}, accV[2] = {zero4, zero4};
    double cE = 0.0, cV = 0.0;  // centre row partial sums
    load(0);
    for (int c = 0; c < Sh::NCH; c++) {
        stage(c);
        // the chunk's fragments, issued before the next chunk's samples
        double f0[Sh::KPC], f1[Sh::KPC];
#pragma unroll
        for (int sl = 0; sl < Sh::KPC; sl++) {
            f0[sl] = tq0[(long)(c * Sh::KPC + sl) * 64];
            f1[sl] = tq1[(long)(c * Sh::KPC + sl) * 64];
        }
        __syncthreads();
        if (c + 1 < Sh::NCH) load(c + 1);  // in flight during this chunk's products
        // every chunk is KPC k-steps of both tables: no branch, so that the operand reads
        // are issued ahead of the products
#pragma unroll
        for (int sl = 0; sl < Sh::KPC; sl++) {
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                accE[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0[sl], bop(0, pm0, sl, ct), accE[ct], 0, 0, 0);
                accV[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0[sl], bop(2, pm0, sl, ct), accV[ct], 0, 0, 0);
            }
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
                accV[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(f1[sl], bop(1, 1 - pm0, sl, ct), accV[ct], 0, 0, 0);
        }
        if (centre) {
            // column tid % 32; of each BASE samples, those of index tid / 32 + HW j, whatever the
            // chunk: the order of this sum is the same in the forms of both chunk lengths
            constexpr int HW = NT / 32, BASE = DShape<FN>::CHK;
            static_assert(!Sh::CENTRE || BASE % CHK == 0, "chunks of one form tile those of the other");
            const int col = tid & 31;
            for (int qq = ((tid >> 5) + HW - c * CHK % BASE % HW) % HW; qq < CHK; qq += HW) {
                const int q = c * CHK + qq;
                const double w0 = ctr[q];
                cE = fma(w0, lds[(0 * CHK + qq) * kCols + col], cE);
                cV = fma(w0, lds[(4 * CHK + qq) * kCols + col], cV);
                cV = fma(ctr[N + 1 + q], lds[(3 * CHK + qq) * kCols + col], cV);
            }
        }
        __syncthreads();  // the operands are read before the next chunk (or the stage) overwrites them
    }
    // output stage [pencil][SR][re, im], one output at a time (N_v, then N_eta): local row
    // j < 16 TPB is p = p0 + j, row 16 TPB + j its mirror N - p, row 32 TPB the centre
    const int p0 = 16 * h * TPB;
    double* out = lds;
    double cen[2] = {0.0, 0.0};  // centre row sums of N_v, N_eta (threads tid < kCols)
    if (centre) {
        cE += __shfl_xor(cE, 32);
        cV += __shfl_xor(cV, 32);
        if (lane < 32) cpart[wave][0][lane] = cE, cpart[wave][1][lane] = cV;
    }
    __syncthreads();
    if (centre && tid < kCols) {
        for (int w = 0; w < 2 * TPB; w++) cen[1] += cpart[w][0][tid], cen[0] += cpart[w][1][tid];
        cen[1] = fma(ctr[N], hN[0][tid], cen[1]);
        cen[0] = fma(ctr[N], hN[2][tid], cen[0]);
    }
    // the centre sample q = N (G+ only): sym rows Q0s[p][N] h3_N, h1_N; anti rows Q1a[p][N] h2_N
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int p = 16 * rt + kq + 4 * r;
        const double w = anti ? (p < Sh::RA ? tab[Sh::COLN_OFF + Sh::RS + p] : 0.0)
                              : (p < Sh::RS ? tab[Sh::COLN_OFF + p] : 0.0);
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            if (anti) {
                accV[ct][r] = fma(w, hN[1][ct * kPencils + lc], accV[ct][r]);
            } else {
                accE[ct][r] = fma(w, hN[0][ct * kPencils + lc], accE[ct][r]);
                accV[ct][r] = fma(w, hN[2][ct * kPencils + lc], accV[ct][r]);
            }
        }
    }
    const int ph = mb.phase[slot];
    const long PS = (long)d.P * nz;
    const long po = ((long)ky0 * d.hnx + kx) * nz, pstride = (long)d.hnx * nz;
#pragma unroll
    for (int o = 0; o < 2; o++) {
        const v4d* acc = o ? accE : accV;
        // sym waves write S to rows p and N - p, then anti waves add A to row p and
        // subtract it from row N - p
        if (!anti) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int j = 16 * wave + kq + 4 * r, p = p0 + j;
                if (p >= Sh::RS || (Sh::CENTRE && p == N / 2)) continue;
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    out[(lc * SR + j) * 2 + ct] = acc[ct][r];
                    out[(lc * SR + 16 * TPB + j) * 2 + ct] = acc[ct][r];
                }
            }
        }
        if (centre && tid < kCols) out[((tid % kPencils) * SR + 32 * TPB) * 2 + tid / kPencils] = cen[o];
        __syncthreads();
        if (anti) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int j = 16 * (wave - TPB) + kq + 4 * r, p = p0 + j;
                if (p >= Sh::RA) continue;
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    out[(lc * SR + j) * 2 + ct] += acc[ct][r];
                    out[(lc * SR + 16 * TPB + j) * 2 + ct] -= acc[ct][r];
                }
            }
        }
        __syncthreads();
        double2* dst = NL + slot * sNL + (o ? 2 + ph : ph) * PS;
        const double2* ov = (const double2*)out;
        for (int i = tid; i < nb * SR; i += NT) {
            const int bb = i / SR, j = i - bb * SR;
            int row;
            if (j < 16 * TPB) {
                const int p = p0 + j;
                row = p < Sh::RS && !(Sh::CENTRE && p == N / 2) ? p : -1;
            } else if (j < 32 * TPB) {
                const int p = p0 + j - 16 * TPB;
                row = p < Sh::RA ? N - p : -1;
            } else {
                row = centre ? N / 2 : -1;
            }
            if (row >= 0) dst[po + bb * pstride + row] = ov[i];
        }
        if (o == 0) __syncthreads();  // the stage is read before N_eta overwrites it
    }
}

// -------------------------------------------------------------------------------------
// The padded p2s of lengths without a compiled plan (any N = nz - 1), as the same kind of FP64
// matrix products with N a run-time number.  The runtime-plan FFT kernel it replaces (k_p2s_nl<0>;
// RPCF_P2S_MFMA=0 keeps it) runs 3 to 5 passes over LDS with index arithmetic by run-time strides:
// 62 us at 40x46x60 (N = 45) against 10.3 here, 281 at 100x151x100 (N = 150, where the product's N^2
// meets the FFT's N log N) against 70.  A chunk's fragments are requested before its samples are
// staged (11.6 against 12.3 us at 40x46x60, 13.9 against 14.5 at 64x61x64; k_p2s_dmfma, with more
// registers held meanwhile, gains nothing by it).  Bound by the latency of a block's phases on small grids, by
// the matrix cores' FP64 rate, operand reads and fragment reads from L2 on long lengths (0.3 of 72
// TFLOP/s, what a large FP64 matrix product reaches, at N = 150).
// -------------------------------------------------------------------------------------
namespace cheb_dmfma {

// Sizes of the products of one N.  Rows of the p2s: sym p <= N/2 (NS), anti p <= (N-1)/2 (NA),
// each in RT row tiles; samples q <= N in NCH chunks of kNChunk.  All tables are zero-padded.
constexpr int kNChunk = 16;
struct NShape {
    int N, NS, NA, RT, NCH, KP;
};
inline NShape nshape(int N) {
    NShape s;
    s.N = N;
    s.NS = N / 2 + 1;
    s.NA = (N + 1) / 2;
    s.RT = ceil_div(s.NS, 16);
    s.NCH = ceil_div(N + 1, kNChunk);
    s.KP = s.NCH * (kNChunk / 4);
    return s;
}
// LDS bytes: the operands [set h3, h2, h1][G+, G-][kNChunk][kCols] or the output rows
// [pencil][nz] of one term
inline size_t p2s_n_lds(const NShape& s) {
    const size_t ops = sizeof(double) * 3 * 2 * kNChunk * kCols, out = sizeof(double2) * kPencils * (s.N + 1);
    return ops > out ? ops : out;
}

// Sizes of the s2p product of one N: RH tiles of the rows 0 < q < N/2; coefficients k = 4j, 4j + 2
// and odd in K0, K2 and K1 k-steps (even counts); CW groups of 16 pencils per block.
struct SShape {
    int N, RH, K0, K2, K1;
};
inline SShape sshape(int N) {
    SShape s;
    s.N = N;
    s.RH = N > 2 ? ceil_div((N - 1) / 2, 16) : 1;
    s.K0 = 2 * ceil_div(N / 4 + 1, 8);
    s.K2 = 2 * ceil_div((N + 2) / 4, 8);
    s.K1 = 2 * ceil_div((N + 1) / 2, 8);
    return s;
}
// A block: CW groups of 8 CT pencils, one wave per row tile and group; where that makes fewer than
// three waves, two more (which take the sums of the special rows meanwhile).
__host__ __device__ inline int s2p_extra(int waves) { return waves < 3 ? 2 : 0; }
inline int s2p_threads(const SShape& s, int cw) { return 64 * (s.RH * cw + s2p_extra(s.RH * cw)); }
// LDS rows of the coefficients: 16 bytes past a multiple of 128, for the writes along k
__host__ __device__ constexpr int s2p_ld(int cw, int ct) { return cw * ct * 16 + 2; }
inline size_t s2p_lds(const SShape& s, int cw, int ct) {
    return sizeof(double) * 4 * (s.K0 + s.K2 + s.K1) * s2p_ld(cw, ct);
}

}  // namespace cheb_dmfma

// Padded p2s + derivative + rhsNonlinear + unpadded s2p (as k_p2s_dmfma), one item a block:
// 2 RT waves, wave w < RT the sym row tile w, the others the anti tiles, each over both column
// tiles.  The centre sample q = N is a sample like the others (G+ = f_N, G- = 0).
template <int RT>
__global__ __launch_bounds__(128 * RT) void k_p2s_dmfma_n(const double2* __restrict__ Z1, long zstride, long sY,
                                                          double2* __restrict__ NL, long sNL, Dims d,
                                                          const double* __restrict__ tab, cheb_dmfma::NShape sh,
                                                          Members mb) {
    using namespace cheb_dmfma;
    constexpr int NT = 128 * RT, UPT = ceil_div(kNChunk * kPencils, NT);
    RPCF_LDS(double);
    const int N = sh.N, nz = N + 1, pz = 2 * N + 1;
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, lc = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool anti = wave >= RT;
    const int rt = anti ? wave - RT : wave;
    const int slot = mb.ids[blockIdx.z], kx = blockIdx.y, ky0 = blockIdx.x * kPencils;
    const int nb = min(kPencils, d.ny - ky0);
    const double2* in = Z1 + slot * sY + (long)kx * pz * d.ny + ky0;
    double2 sa[UPT][3], sb[UPT][3];
    auto load = [&](int c) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int i = tid + u * NT, q = c * kNChunk + i / kPencils, b = i % kPencils;
            const bool ok = i < kNChunk * kPencils && q <= N && b < nb;
            const long oa = ok ? (long)q * d.ny + b : 0, ob = ok ? (long)(2 * N - q) * d.ny + b : 0;
#pragma unroll
            for (int g = 0; g < 3; g++) {
                sa[u][g] = in[g * zstride + oa];
                sb[u][g] = in[g * zstride + ob];
            }
        }
    };
    load(0);  // before anything waits on memory
    const double aphi = mb.mp[slot].aphi, beta = mb.mp[slot].beta;
    auto stage = [&](int c) {
#pragma unroll
        for (int u = 0; u < UPT; u++) {
            const int i = tid + u * NT;
            if (i >= kNChunk * kPencils) continue;
            const int qq = i / kPencils, b = i % kPencils, q = c * kNChunk + qq, ky = ky0 + b;
            const double ia = (double)kx / aphi;
            const double ib = ky >= d.ny / 2 + 1 ? (double)(ky - d.ny) / beta : (double)ky / beta;
            const double k2 = ia * ia + ib * ib;
            const bool mean = kx == 0 && ky == 0, ok = b < nb && q <= N;
#pragma unroll
            for (int pm = 0; pm < 2; pm++) {
                double2 f[3];
#pragma unroll
                for (int g = 0; g < 3; g++) {
                    const double2 a = sa[u][g], m = sb[u][g];
                    f[g] = pm ? make_double2(a.x - m.x, a.y - m.y) : make_double2(a.x + m.x, a.y + m.y);
                    if (q == N) f[g] = pm ? make_double2(0.0, 0.0) : a;
                    if (!ok) f[g] = make_double2(0.0, 0.0);
                }
                const double2 x = f[0], y = f[1], z = f[2];
                const double2 h3 = mean ? y : make_double2(-ia * y.y + ib * x.y, ia * y.x - ib * x.x);
                const double2 h2 = mean ? make_double2(0.0, 0.0)
                                        : make_double2(-ia * x.y - ib * y.y, ia * x.x + ib * y.x);
                const double2 h1 = mean ? x : make_double2(k2 * z.x, k2 * z.y);
                double* o = lds + (pm * kNChunk + qq) * kCols + b;
                o[0] = h3.x;
                o[kPencils] = h3.y;
                o[2 * kNChunk * kCols] = h2.x;
                o[2 * kNChunk * kCols + kPencils] = h2.y;
                o[4 * kNChunk * kCols] = h1.x;
                o[4 * kNChunk * kCols + kPencils] = h1.y;
            }
        }
    };
    // tables Q0s, Q0a, Q1s, Q1a, [RT][KP] fragments each: sym waves Q0 = Q0s over G+ (h3, h1),
    // Q1 = Q1s over G- (h2); anti waves Q0a over G-, Q1a over G+
    const long tsz = (long)RT * sh.KP * 64;
    const double* tq0 = tab + (anti ? tsz : 0) + (long)rt * sh.KP * 64 + lane;
    const double* tq1 = tq0 + 2 * tsz;
    const int pm0 = anti ? 1 : 0;
    auto bop = [&](int set, int pm, int sl, int ct) {
        return lds[((set * 2 + pm) * kNChunk + 4 * sl + kq) * kCols + ct * kPencils + lc];
    };
    const v4d zero4 = {0.0, 0.0, 0.0, 0.0};
    v4d accE[2] = {zero4, zero4}, accV[2] = {zero4, zero4};
    for (int c = 0; c < sh.NCH; c++) {
        // the chunk's fragments, in flight while its samples are staged
        double f0[kNChunk / 4], f1[kNChunk / 4];
#pragma unroll
        for (int sl = 0; sl < kNChunk / 4; sl++) {
            f0[sl] = tq0[(long)(c * (kNChunk / 4) + sl) * 64];
            f1[sl] = tq1[(long)(c * (kNChunk / 4) + sl) * 64];
        }
        stage(c);
        __syncthreads();
        if (c + 1 < sh.NCH) load(c + 1);
#pragma unroll
        for (int sl = 0; sl < kNChunk / 4; sl++)
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                accE[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0[sl], bop(0, pm0, sl, ct), accE[ct], 0, 0, 0);
                accV[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0[sl], bop(2, pm0, sl, ct), accV[ct], 0, 0, 0);
                accV[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(f1[sl], bop(1, 1 - pm0, sl, ct), accV[ct], 0, 0, 0);
            }
        __syncthreads();  // the operands are read before the next chunk or the output overwrites them
    }
    // sym waves write S to rows p and N - p, then the anti waves add and subtract A
    const int ph = mb.phase[slot];
    const long PS = (long)d.P * nz, po = ((long)ky0 * d.hnx + kx) * nz, pstride = (long)d.hnx * nz;
    double* out = lds;
#pragma unroll
    for (int o = 0; o < 2; o++) {
        const v4d* acc = o ? accE : accV;
#pragma unroll
        for (int half = 0; half < 2; half++) {
            if ((half == 1) == anti) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int p = 16 * rt + kq + 4 * r;
                    if (p >= (anti ? sh.NA : sh.NS)) continue;
#pragma unroll
                    for (int ct = 0; ct < 2; ct++) {
                        double* a = out + (lc * nz + p) * 2 + ct;
                        double* m = out + (lc * nz + N - p) * 2 + ct;
                        if (anti) *a += acc[ct][r], *m -= acc[ct][r];
                        else *a = acc[ct][r], *m = acc[ct][r];
                    }
                }
            }
            __syncthreads();
        }
        double2* dst = NL + slot * sNL + (o ? 2 + ph : ph) * PS;
        const double2* ov = (const double2*)out;
        for (int bb = wave; bb < nb; bb += 2 * RT)
            for (int j = lane; j < nz; j += 64) dst[po + bb * pstride + j] = ov[bb * nz + j];
        if (o == 0) __syncthreads();
    }
}

// Padded s2p of the FP64 form: F[6][P][nz] -> Y[6][kx][q][ky], f_q = sum_k a_k cos(pi k q/(2N)),
// as dense products on the matrix cores.  The cosines fold twice: with E0, E2 and O the sums over
// k = 4j, k = 4j + 2 and odd k at row q, and O' that over odd k at row N - q,
//   f_q = E0 + E2 + O, f_{N-q} = E0 - E2 + O', f_{N+q} = E0 - E2 - O', f_{2N-q} = E0 + E2 - O
// so the rows 0 < q < N/2 give all the others, for 3/4 N^2 products a column; the rows 0, N, 2N and
// N/2, 3N/2 (N even) are sums on the vector units.  A block takes CW groups of pencils of a field,
// their coefficients in LDS as B operands, with one wave per row tile and group; the fragments
// stream from L2, two k-step pairs ahead, and the rows leave from the accumulators.  A group is 16
// pencils (CT = 2: a tile of their real parts and one of their imaginary parts, 256 contiguous
// bytes of a row), or on small grids 8 (CT = 1: real and imaginary parts share a tile), whose
// waves run half as many products each.  Bound by the latency of a block's phases on small grids,
// by memory, the fragments' reads from L2 and the matrix cores' rate (N^2) on large ones: 233 us at
// 256x97x256 (the bytes take 188 at the copy rate), 90 at 128x129x128 (63), 40 at 128x65x128, 16.3
// at 64x65x64, 7.6 at 32x33x32; the half-length FFTs of k_cheb_s2p_h take 274, 97, 56, 22.9 and
// 10.3.  With the first fold only (N^2 products) it took 360 at 256x101x256 and 107 at 128x126x128,
// now 273 and 85.  96 registers keep five waves a SIMD: with four, 265 at 256x97x256.
template <int CT>
__global__ __launch_bounds__(512, 5) void k_s2p_dmfma(const double2* __restrict__ F, long fstride, long sF,
                                                   double2* __restrict__ Y, long ystride, long sY, Dims d,
                                                   const double* __restrict__ tab, cheb_dmfma::SShape sh, int CW,
                                                   const int* __restrict__ ids) {
    using namespace cheb_dmfma;
    RPCF_LDS(double);
    constexpr int G = 8 * CT;  // pencils per group; columns [group][re, im][pencil]
    const int N = sh.N, nz = N + 1, pz = 2 * N + 1, ld = s2p_ld(CW, CT), nthr = blockDim.x;
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, lc = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rt = wave % sh.RH, cg = wave / sh.RH;
    const int f = blockIdx.z % 6, kx = blockIdx.y, ky0 = blockIdx.x * G * CW;
    const long slot = ids[blockIdx.z / 6];
    const int nb = min(G * CW, d.ny - ky0);
    const double2* in = F + slot * sF + f * fstride + ((long)ky0 * d.hnx + kx) * nz;
    double2* out = Y + slot * sY + f * ystride + (long)kx * pz * d.ny + ky0;
    const int rows0 = 4 * sh.K0, rows2 = 4 * sh.K2, rows = rows0 + rows2 + 4 * sh.K1;
    // coefficient k of pencil b to its set's row; zeros in the rows past the coefficients
    {
        const FastDiv by_nz(nz);
        const int pstride = d.hnx * nz;
        staged<8>(
            G * CW * nz, tid, nthr,
            [&](int i) {
                const unsigned b = (unsigned)i / by_nz, k = i - b * nz;
                return (int)b < nb ? in[b * pstride + k] : make_double2(0.0, 0.0);
            },
            [&](int i, double2 v) {
                const unsigned b = (unsigned)i / by_nz, k = i - b * nz;
                const unsigned r = k & 1 ? rows0 + rows2 + (k >> 1) : k & 2 ? rows0 + (k >> 2) : k >> 2;
                double* o = lds + r * ld + (b / G) * (2 * G) + b % G;
                o[0] = v.x;
                o[G] = v.y;
            });
        for (int i = tid; i < (rows - nz) * 2 * G * CW; i += nthr) {
            int r = i / (2 * G * CW);
            const int c = i - r * 2 * G * CW;
            const int n0 = N / 4 + 1, n2 = (N + 2) / 4;
            if (r < rows0 - n0) r += n0;
            else if ((r -= rows0 - n0) < rows2 - n2) r += rows0 + n2;
            else r += -(rows2 - n2) + rows0 + rows2 + (N + 1) / 2;
            lds[r * ld + c] = 0.0;
        }
    }
    __syncthreads();
    const int P0 = sh.K0 / 2, P2 = P0 + sh.K2 / 2, P1 = P2 + sh.K1 / 2;  // ends of the sets in k-step pairs
    const v4d zero4 = {0.0, 0.0, 0.0, 0.0};
    v4d e0[CT], e2[CT], o1[CT], om[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++) e0[ct] = e2[ct] = o1[ct] = om[ct] = zero4;
    if (cg < CW) {
        const double* t = tab + (long)rt * (sh.K0 + sh.K2 + 2 * sh.K1) * 64 + lane;
        const double* tm = t + (sh.K0 + sh.K2 + sh.K1) * 64;
        const double* bl = lds + kq * ld + cg * 16 * CT + lc;
        double c0 = t[0], c1 = t[64], n0 = t[128 * min(1, P1 - 1)], n1 = t[128 * min(1, P1 - 1) + 64];
        double m0 = tm[0], m1 = tm[64];
        auto pairs = [&](int p, int end, v4d* acc, bool mirror) {
            for (; p < end; p++) {
                const int nx = 128 * min(p + 2, P1 - 1), mx = 128 * min(max(p + 1 - P2, 0), P1 - P2 - 1);
                const double f0 = t[nx], f1 = t[nx + 64];
                const double* b = bl + 8 * p * ld;
                double b0[CT], b1[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ct++) b0[ct] = b[16 * ct], b1[ct] = b[4 * ld + 16 * ct];
#pragma unroll
                for (int ct = 0; ct < CT; ct++) acc[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(c0, b0[ct], acc[ct], 0, 0, 0);
                if (mirror) {
                    const double g0 = tm[mx], g1 = tm[mx + 64];
#pragma unroll
                    for (int ct = 0; ct < CT; ct++) om[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(m0, b0[ct], om[ct], 0, 0, 0);
#pragma unroll
                    for (int ct = 0; ct < CT; ct++) om[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(m1, b1[ct], om[ct], 0, 0, 0);
                    m0 = g0, m1 = g1;
                }
#pragma unroll
                for (int ct = 0; ct < CT; ct++) acc[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(c1, b1[ct], acc[ct], 0, 0, 0);
                c0 = n0, c1 = n1, n0 = f0, n1 = f1;
            }
        };
        pairs(0, P0, e0, false);
        pairs(P0, P2, e2, false);
        pairs(P2, P1, o1, true);
    }
    const int bp = cg * G + (CT == 2 ? lc : lc & 7);  // this lane's pencil
    if (cg < CW && bp < nb) {
        // CT = 2: (re, im) of a row; CT = 1: the part of this lane
        double* o = (double*)(out + bp) + (CT == 2 ? 0 : lc >> 3);
        const long ny = 2 * d.ny;
        auto put = [&](long q, double x, double y) {
            if constexpr (CT == 2) *(double2*)(o + q * ny) = make_double2(x, y);
            else o[q * ny] = x;
        };
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int q = 1 + 16 * rt + kq + 4 * r;
            if (2 * q >= N) continue;
            constexpr int I = CT - 1;
            const double s0 = e0[0][r] + e2[0][r], s1 = e0[I][r] + e2[I][r];
            const double t0 = e0[0][r] - e2[0][r], t1 = e0[I][r] - e2[I][r];
            put(q, s0 + o1[0][r], s1 + o1[I][r]);
            put(N - q, t0 + om[0][r], t1 + om[I][r]);
            put(N + q, t0 - om[0][r], t1 - om[I][r]);
            put(2 * N - q, s0 - o1[0][r], s1 - o1[I][r]);
        }
    }
    // rows 0, N, 2N: sums of the three sets; rows N/2, 3N/2: k = 4j with signs (-1)^j, odd k with
    // cos(pi k/4).  A wave takes 16 columns, a quarter of the coefficients a lane.
    const int extra = s2p_extra(sh.RH * CW), waves = nthr >> 6, first = extra ? sh.RH * CW : 0;
    for (int task = wave - first; task < CT * CW; task += waves - first) {
        if (task < 0) break;
        const int c = 16 * task + lc, b = c / (2 * G) * G + c % G, im = c / G & 1;
        const double* col = lds + c;
        double s0 = 0.0, s2 = 0.0, s1 = 0.0, z0 = 0.0, z1 = 0.0;
#pragma unroll 4
        for (int r = kq; r < rows0; r += 4) {
            const double v = col[r * ld];
            s0 += v;
            z0 += kq & 1 ? -v : v;
        }
#pragma unroll 4
        for (int r = kq; r < rows2; r += 4) s2 += col[(rows0 + r) * ld];
#pragma unroll 4
        for (int r = kq; r < rows - rows0 - rows2; r += 4) {
            const double v = col[(rows0 + rows2 + r) * ld];
            s1 += v;
            z1 += (kq + 1) & 2 ? -v : v;
        }
#pragma unroll
        for (int m = 16; m <= 32; m *= 2) {
            s0 += __shfl_xor(s0, m), s2 += __shfl_xor(s2, m), s1 += __shfl_xor(s1, m);
            z0 += __shfl_xor(z0, m), z1 += __shfl_xor(z1, m);
        }
        if (b >= nb) continue;
        double* o = (double*)(out + b) + im;
        const long ny = 2 * d.ny;
        z1 *= 0.70710678118654752440;
        if (kq == 0) o[0] = s0 + s2 + s1;
        else if (kq == 1) o[N * ny] = s0 - s2;
        else if (kq == 2) o[2 * N * ny] = s0 + s2 - s1;
        else if (!(N & 1)) {
            o[N / 2 * ny] = z0 + z1;
            o[(N + N / 2) * ny] = z0 - z1;
        }
    }
}
