// dg_cnn.hip -- kernels of the learned conservative flux correction.
//
// The network is a 3D CNN 5 -> 32 -> 32 -> 15 (3x3x3 kernels, GELU after the
// first two layers): from the primitive state of a grid it predicts, for
// each cell c and axis d, a correction to the five flux components on the
// face c + e_d/2.  Convolutions run on MFMA (bf16 operands, fp32
// accumulation) as implicit GEMMs:
//
//   forward / input-gradient  D[cout][cell] = sum_k W[k][cout] * X[cell, k],
//                             k = tap * CIN + cin, tap = (dx*3 + dy)*3 + dz;
//                             A = weights (pre-packed in MFMA fragment order,
//                             held in VGPRs), B = activations (channels-last)
//                             read from input planes in LDS, 16 B per lane
//                             and k-step (conv_ring_kernel);
//   weight gradient           D[cout][k] = sum_cells dZ[cell][cout] * X[cell + tap][cin],
//                             both operands channels-last in LDS, transposed
//                             by the LDS reads (dw_kernel); one partial per
//                             workgroup, reduced in a fixed order.
//
// MFMA lane layouts (gfx950):
//   v_mfma_f32_32x32x16_bf16: A lane l holds row l%32, k = 8*(l/32) + i;
//     B lane l holds column l%32, same k; D lane l holds column l%32,
//     rows 8*(i/4) + 4*(l/32) + i%4 for its 16 values i.
//   v_mfma_f32_16x16x32_bf16: A lane l holds row l%16, k = 8*(l/16) + i;
//     B lane l holds column l%16, same k; D lane l holds column l%16,
//     rows 4*(l/16) + i for its 4 values i.
//
// Geometry: convolutions map an input box of (in0, in1, in2) cells per batch
// item to an output box; "valid" (PAD 0) reads in[o + d], out = in - 2;
// "full" (PAD 2, the input gradient) reads in[o + d - 2] with zeros outside,
// out = in + 2.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "dg_cnn.h"

namespace dg {
namespace cnn {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------- helpers --
// GELU(z) = z Phi(z) = 0.5 z (1 + erf(z / sqrt 2)), with erf from Abramowitz &
// Stegun 7.1.26 (rational approximation in t = 1 / (1 + p|x|) times exp(-x^2),
// absolute error <= 1.5e-7, far below the bf16 rounding of the activations):
// one reciprocal and one exp2 instead of a library erff.
struct ErfExp {
    float erf, e;   // erf(x), exp(-x^2)
};
__device__ __forceinline__ ErfExp erf_as(float x)
{
    const float ax = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, ax, 1.0f));
    const float e = __builtin_amdgcn_exp2f(-1.44269504088896341f * x * x);   // (a denormal one is zero)
    float p = fmaf(1.061405429f, t, -1.453152027f);
    p = fmaf(p, t, 1.421413741f);
    p = fmaf(p, t, -0.284496736f);
    p = fmaf(p, t, 0.254829592f);
    p *= t;
    return {copysignf(fmaf(-p, e, 1.0f), x), e};
}
__device__ __forceinline__ float gelu(float z)
{
    const float h = 0.5f * z;
    return fmaf(h, erf_as(z * 0.70710678118654752f).erf, h);
}
// GELU'(z) = Phi(z) + z phi(z), phi(z) = exp(-z^2 / 2) / sqrt(2 pi)
__device__ __forceinline__ float gelu_grad(float z)
{
    const ErfExp r = erf_as(z * 0.70710678118654752f);
    return fmaf(0.5f, r.erf, 0.5f) + z * 0.39894228040143268f * r.e;
}

// 32-bit integer hash (xorshift-multiply finalizer)
__device__ __forceinline__ uint32_t mix32(uint32_t x)
{
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

__device__ __forceinline__ bf16x8 zero8()
{
    bf16x8 v;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (bf16)0.0f;
    return v;
}

// As convolutions the layers use v_mfma_f32_16x16x32_bf16: a k-step is 32
// consecutive k of one x tap, i.e. TPS (y, z) taps of all CIN channels, and a
// wave computes 16 of the COUT output channels.
template <int CIN, int COUT> struct ConvCfg {
    static constexpr int TPS = 32 / CIN;               // (y, z) taps per k-step
    static constexpr int KS = (9 + TPS - 1) / TPS;     // k-steps per input plane
    static constexpr int CG = COUT / 16;               // groups of output channels
    static constexpr int WAVES = CIN == 8 ? 16 : 8;    // one workgroup per CU
    static constexpr int EU = WAVES / 4, THREADS = 64 * WAVES;
    static constexpr int NT = 16 * CG / WAVES;         // 16-cell tiles per wave (256 cells per workgroup)
    // 32 -> 32 has the registers for 2 activation fragments in flight and for half
    // of a thread's share of the next plane at a time, 16 -> 32 for half a share;
    // otherwise they spill (204 us instead of 155)
    static constexpr int DEPTH = KS * NT == 36 ? 2 : 4, PARTS = CIN == 16 || KS * NT == 36 ? 2 : 1;
};

// ---------------------------------------------------------- conv (MFMA) --
// EPI_TRAIN: Z = acc + b (fp32 out), X = bf16(gelu(Z));  EPI_INFER: X only;
// EPI_OUT: Y = acc + b (fp32, COUT channels);  EPI_BWD: X = bf16(acc * gelu'(Zprev));
// EPI_OUT16: X = bf16(acc + b) (the output layer for the learned step's correction).
enum { EPI_TRAIN = 0, EPI_INFER = 1, EPI_OUT = 2, EPI_BWD = 3, EPI_OUT16 = 4 };

// --------------------------------------------- conv (MFMA, LDS planes) --
// The same convolutions with the activations staged in LDS.  A workgroup owns
// a rectangle of ry x rz output (y, z) positions, flattened row-major (at most
// 256 in tiles of 16, split over the waves; with 32 output channels a wave takes
// 16 of them), and marches the INPUT planes of a chunk along
// x.  Input plane j feeds the output planes j, j - 1 and j - 2 (x taps 0, 1,
// 2), whose accumulators are all in registers: every activation fragment read
// from LDS is used by three MFMAs, and only two plane slots are needed, one
// read while the next plane is loaded to registers (before the MFMAs) and
// stored (after them), one barrier per plane.  A slot holds (ry + 2) rows of
// RING_ROWP cells; a cell is CIN bf16 channels in 16-B chunks, padded by one
// chunk for CIN >= 16 so that the 128-bit reads of consecutive cells hit
// distinct banks.  Cells outside the input box load zeros (the full
// convolution's padding).  The weights stay in VGPRs.
// Two waves per SIMD (four with CIN 8) run the matrix cores under each other's
// epilogues; the epilogue of a finished plane (GELU) is spread one value at a
// time over the next plane's k-steps.  Bound by instruction issue: an MFMA
// keeps the SIMD's VALU from issuing for some 10 of its 16 cycles, and with 32
// outputs the epilogues take as long as the MFMAs.  An activation fragment per
// MFMA (outputs gathered from four slots, one wave per SIMD), as before, was
// bound by LDS and overlapped nothing.  Learned step of 128^3, layers 1-3: 124,
// 204, 126 -> 85, 155, 59 us; training batch of 8 crops of 32^3, layers 1-3
// forward 39, 47, 30 -> 25, 31, 17, input gradients of layers 2 and 3 80, 39 ->
// 50, 30.
constexpr int RING_POS = 256;               // output positions per workgroup plane
constexpr int RING_ROWP = 48;               // cells per LDS row: rz + 2 <= RING_ROWP
constexpr int RING_RMAX = 10;               // LDS rows per slot: ry + 2 <= RING_RMAX

struct RingGeom {
    ConvGeom g;
    int ry, rz;        // output rectangle of a workgroup: ry * rz <= RING_POS
    int ny, nz;        // rectangles along y, z
    int cx, nxc;       // output planes per work item, chunks along x
    long long items;   // B * nxc * ny * nz
};

template <int CIN> struct RingCell {
    static constexpr int NC = CIN / 8;                   // 16-B chunks of channels per cell
    static constexpr int CS = NC == 1 ? 1 : NC + 1;      // chunk stride of a cell
    static constexpr int SLOT = RING_RMAX * RING_ROWP * CS * 16;   // bytes per slot
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// zeros for the cells outside the input box (never written)
static __device__ __attribute__((aligned(16))) uint32_t ring_zero[4];

// Computed here: an index of which no 64-bit address is kept across the planes,
// or a value that is not sunk into the branch that stores it.
template <typename T> __device__ __forceinline__ T opaque(T v)
{
#ifdef __AMDGCN__
    asm volatile("" : "+v"(v));
#endif
    return v;
}

template <int CIN, int COUT, int EPI, int PAD>
__global__ void __launch_bounds__((ConvCfg<CIN, COUT>::THREADS))
    __attribute__((amdgpu_waves_per_eu((ConvCfg<CIN, COUT>::EU), (ConvCfg<CIN, COUT>::EU))))
conv_ring_kernel(const RingGeom rg, const bf16 *__restrict__ X, const bf16x8 *__restrict__ Wp,
                 const float *__restrict__ bias, float *__restrict__ Zout, bf16 *__restrict__ Xout,
                 float *__restrict__ Yout, const float *__restrict__ Zprev)
{
    typedef ConvCfg<CIN, COUT> C;
    typedef RingCell<CIN> RC;
    constexpr int NT = C::NT, KS = C::KS;
    __shared__ __attribute__((aligned(16))) char ring[2 * RC::SLOT];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cg = wave % C::CG, pg = wave / C::CG;
    const int col = lane & 15, part = lane >> 4;
    const ConvGeom &g = rg.g;

    bf16x8 wa[KS][3];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) wa[s][dx] = Wp[((cg * KS + s) * 3 + dx) * 64 + lane];
    const int ch = 16 * cg + 4 * part;   // this lane's four output channels
    f32x4 bv = {0, 0, 0, 0};             // their biases: the sums start there
    if (EPI != EPI_BWD) bv = *reinterpret_cast<const f32x4 *>(bias + ch);
    // byte offset of this lane's 8 channels of k-step s from its cell: with CIN 32
    // a constant, with less the lane groups read different taps (past the last:
    // that one again, with zero weights)
    int po[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int tap = C::TPS == 1 ? s : min(s * C::TPS + part / RC::NC, 8);
        po[s] = (tap / 3 * RING_ROWP + tap % 3) * RC::CS * 16;
    }

    const int RY = rg.ry, RZ = rg.rz, npos = RY * RZ;
    const int o0 = g.out[0], o1 = g.out[1], o2 = g.out[2];
    for (long long item = blockIdx.x; item < rg.items; item += gridDim.x) {
        long long r = item;
        const int iz = (int)(r % rg.nz); r /= rg.nz;
        const int iy = (int)(r % rg.ny); r /= rg.ny;
        const int xc = (int)(r % rg.nxc);
        const int b = (int)(r / rg.nxc);
        const int y0 = iy * RY, z0 = iz * RZ;
        const int xs = xc * rg.cx, n = min(rg.cx, o0 - xs);   // output planes of the item

        // this lane's positions: LDS byte offset (of the plane's slot), output (y, z) index
        int lb[NT], oyz[NT];
        bool ok[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int p = (pg * NT + t) * 16 + col;
            const int pp = p < npos ? p : 0;
            const int py = pp / RZ, pz = pp - py * RZ;
            ok[t] = p < npos && y0 + py < o1 && z0 + pz < o2;
            lb[t] = ((py * RING_ROWP + pz) * RC::CS + part % RC::NC) * 16;
            oyz[t] = ok[t] ? (y0 + py) * o2 + z0 + pz : 0;
        }

        // Staging of an input plane: each thread loads its 16-B chunks to registers
        // and stores them after the plane's MFMAs (PARTS 2: in halves, each after
        // half of them).  off: chunk in the plane, -1 for zeros (outside the box, or
        // cells that no output needs).
        constexpr int CHUNKS = RING_RMAX * RING_ROWP * RC::NC, PER = (CHUNKS + C::THREADS - 1) / C::THREADS;
        static_assert(C::THREADS % RC::NC == 0, "a thread's chunks are one channel group");
        constexpr int PARTS = C::PARTS, PART = (PER + PARTS - 1) / PARTS;
        u32x4 fv[PART];
        int off[PER];
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int cell = (k * C::THREADS + (int)threadIdx.x) / RC::NC, fy = cell / RING_ROWP, fz = cell % RING_ROWP;
            const int yi = y0 - PAD + fy, zi = z0 - PAD + fz;
            const bool in = fy < RY + 2 && fz < RZ + 2 && yi >= 0 && yi < g.in[1] && zi >= 0 && zi < g.in[2];
            off[k] = in ? (yi * g.in[2] + zi) * RC::NC + (int)threadIdx.x % RC::NC : -1;
        }
        auto load_part = [&](int j, int h) {
            const int xi = xs + j - PAD;
            const bool xin = xi >= 0 && xi < g.in[0];
            const u32x4 *src = reinterpret_cast<const u32x4 *>(X) +
                               ((long long)b * g.in[0] + (xin ? xi : 0)) * g.in[1] * g.in[2] * RC::NC;
#pragma unroll
            for (int k = h * PART; k < PER && k < (h + 1) * PART; ++k) {
                const int o = opaque(off[k]);
                fv[k - h * PART] = *(xin && o >= 0 ? src + o : reinterpret_cast<const u32x4 *>(ring_zero));
            }
        };
        const int dst = ((int)threadIdx.x / RC::NC * RC::CS + (int)threadIdx.x % RC::NC) * 16;
        auto store_part = [&](int j, int h) {
            char *slot = ring + (j & 1) * RC::SLOT + dst;
#pragma unroll
            for (int k = h * PART; k < PER && k < (h + 1) * PART; ++k)
                if ((k + 1) * C::THREADS <= CHUNKS || k * C::THREADS + (int)threadIdx.x < CHUNKS)
                    *reinterpret_cast<u32x4 *>(slot + k * (C::THREADS / RC::NC * RC::CS * 16)) = fv[k - h * PART];
        };
#pragma unroll
        for (int h = 0; h < PARTS; ++h) {
            load_part(0, h);
            store_part(0, h);
        }
        __syncthreads();

        // accumulators of the output planes j (0), j - 1 (1) and j - 2 (2); prv:
        // the plane finished before, its epilogue pending
        f32x4 acc[3][NT], prv[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[0][t] = acc[1][t] = acc[2][t] = prv[t] = f32x4{0, 0, 0, 0};
        const long long plane_cells = (long long)o1 * o2;
        const long long mb0 = ((long long)b * o0 + xs) * plane_cells;

        // value q of tile t of the pending plane (output index mb of y = z = 0); the
        // last of a tile stores its four
        float ev[4];
        f32x4 zp[2];   // EPI_BWD: gelu' arguments of this tile and the next
        auto load_z = [&](long long mb, int t) {
            if (EPI == EPI_BWD && t < NT)
                zp[t & 1] = *reinterpret_cast<const f32x4 *>(Zprev + (mb + opaque(oyz[t])) * COUT + ch);
        };
        auto epilogue = [&](long long mb, int t, int q) {
            if (q == 0) load_z(mb, t + 1);
            const float v = EPI == EPI_BWD ? prv[t][q] * gelu_grad(zp[t & 1][q]) : prv[t][q] + bv[q];
            if (EPI == EPI_TRAIN) prv[t][q] = v;
            ev[q] = opaque(EPI == EPI_TRAIN || EPI == EPI_INFER ? gelu(v) : v);
            if (q != 3 || !ok[t]) return;
            const long long m = mb + opaque(oyz[t]);
            if (EPI == EPI_TRAIN) *reinterpret_cast<f32x4 *>(Zout + m * COUT + ch) = prv[t];
            if (EPI == EPI_OUT) {
                *reinterpret_cast<f32x4 *>(Yout + m * COUT + ch) = f32x4{ev[0], ev[1], ev[2], ev[3]};
            } else {
                bf16x4 xo;
#pragma unroll
                for (int i = 0; i < 4; ++i) xo[i] = (bf16)ev[i];
                *reinterpret_cast<bf16x4 *>(Xout + m * COUT + ch) = xo;
            }
        };

        // Input plane j with the x taps of MASK; PENDING: the epilogue of output
        // plane j - 3 along with it.
        auto plane = [&](auto mask, auto pending, int j) {
            constexpr int MASK = decltype(mask)::value;
            constexpr bool PENDING = decltype(pending)::value;
            const bool more = j < n + 1;
            const long long mb = mb0 + (long long)(j - 3) * plane_cells;
            if (PENDING) load_z(mb, 0);
            if (more) load_part(j + 1, 0);
            constexpr int STEPS = KS * NT;
            constexpr int VPS = (4 * NT + STEPS - 1) / STEPS;        // epilogue values per step,
            constexpr int EVERY = VPS > 1 ? 1 : STEPS / (4 * NT);    // or steps per value
            auto load_b = [&](int f) {
                return *reinterpret_cast<const bf16x8 *>(ring + lb[f % NT] + po[f / NT]);
            };
            bf16x8 bq[C::DEPTH];
#pragma unroll
            for (int f = 0; f < C::DEPTH; ++f) bq[f] = load_b(f);
#pragma unroll
            for (int f = 0; f < STEPS; ++f) {
                const int s = f / NT, t = f % NT;
                const bf16x8 bf = bq[f % C::DEPTH];
#pragma unroll
                for (int dx = 2; dx >= 0; --dx)
                    if (MASK >> dx & 1) {
                        const f32x4 c = s ? acc[dx][t] : dx ? acc[dx - 1][t] : f32x4{0, 0, 0, 0};
                        acc[dx][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa[s][dx], bf, c, 0, 0, 0);
                    }
                if (f + C::DEPTH < STEPS) bq[f % C::DEPTH] = load_b(f + C::DEPTH);
                if (PENDING && f % EVERY == 0)
#pragma unroll
                    for (int v = f / EVERY * VPS; v < (f / EVERY + 1) * VPS; ++v)
                        if (v < 4 * NT) epilogue(mb, v / 4, v % 4);
                __builtin_amdgcn_sched_barrier(0);
                if (PARTS == 2 && f == STEPS / 2 && more) {   // the other slot is free since the last barrier
                    store_part(j + 1, 0);
                    load_part(j + 1, 1);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                prv[t] = acc[2][t];
                lb[t] += j & 1 ? -RC::SLOT : RC::SLOT;
            }
            if (more) store_part(j + 1, PARTS - 1);
            __syncthreads();
        };
        typedef std::integral_constant<bool, true> yes;
        typedef std::integral_constant<bool, false> no;
        if (n > 2) {
            plane(std::integral_constant<int, 1>{}, no{}, 0);
            plane(std::integral_constant<int, 3>{}, no{}, 1);
            plane(std::integral_constant<int, 7>{}, no{}, 2);
            for (int j = 3; j < n; ++j) plane(std::integral_constant<int, 7>{}, yes{}, j);
            plane(std::integral_constant<int, 6>{}, yes{}, n);
            plane(std::integral_constant<int, 4>{}, yes{}, n + 1);
        } else {   // x taps without an output plane accumulate in registers that nothing reads
            for (int j = 0; j < 3; ++j) plane(std::integral_constant<int, 7>{}, no{}, j);
            if (n == 2) plane(std::integral_constant<int, 4>{}, yes{}, 3);
        }
        load_z(mb0 + (n - 1) * plane_cells, 0);
#pragma unroll
        for (int v = 0; v < 4 * NT; ++v) epilogue(mb0 + (n - 1) * plane_cells, v / 4, v % 4);
    }
}

// ----------------------------------------------------- weight gradient --
// dW[tap][cin][cout] = sum over the cells of a valid convolution of
// dZ[cell][cout] * X[cell + tap][cin], and db[cout] = sum of dZ, as an MFMA
// GEMM with K = cells: A = dZ^T (32 output channels), B = X at one tap (32
// input channels of a tile; with CIN 8 four taps of 8) or ones (the tap after
// the last, whose columns are the bias gradient).
//
// Both operands need 8 consecutive cells of one channel per lane, but the
// activations are channels-last.  They stay so in LDS, and
// ds_read_b64_tr_b16 transposes on the way to the registers: 16 lanes read 4
// cells x 16 channels, lane i receives channel i of the 4 cells, and since
// every cell has its own address a tap is an offset like any other.
// A workgroup owns a rectangle of ry x rz outputs in (y, z) and marches along
// x over a chunk of planes: a ring of 4 input planes (rows of 48 cells, so
// that taps are constant offsets) and 2 dZ planes, the next ones loaded to
// registers before a plane's MFMAs and stored after them (one barrier per
// plane).  The 28 column tiles (7 with CIN 8) are 7 per wave, held in the
// accumulators to the end: TG waves split the tiles and KG split the cells
// (16 per MFMA); the KG sums are added in LDS in a fixed order and each
// workgroup writes one partial (deterministic).
// Bound by LDS: 8 KB of transposed reads per 7 MFMAs and wave, and the
// staging.  A training batch of 8 crops of 32^3: layers 1-3 in 22, 39 and 35
// us; before, staged channel-major with 2-byte writes and gathered with eight
// 2-byte reads per MFMA, 113, 220 and 200 us, and 41 us for each layer's
// separate bias sums (the Adam step 1.08 -> 0.50 ms).
constexpr int DW_WAVES = 8;
constexpr int DW_ROWP = 48, DW_RMAX = 9;                     // LDS rows of 48 cells, at most 9
constexpr int DW_POS = (DW_RMAX - 2) * (DW_ROWP - 2);        // outputs per rectangle and plane
constexpr int DW_ZCELLS = (DW_POS + 15) / 16 * 16;

struct DwGeom {
    ConvGeom g;
    int ry, rz, magic;   // rectangle; cell / rz == cell * magic >> 16
    int ny, nz;          // rectangles along y, z
    int cx, nxc;         // output planes per work item, chunks along x
    long long items;
};

template <int CIN, int COUT> struct DwCfg {
    static constexpr int XB = CIN * 2, ZB = COUT * 2;        // bytes per cell
    static constexpr int XSLOT = DW_RMAX * DW_ROWP * XB, ZSLOT = DW_ZCELLS * ZB;
    static constexpr int NTILES = 28 * CIN / 32;
    static constexpr int TPW = 7, TG = NTILES / TPW, KG = DW_WAVES / TG;
    static constexpr int STAGE = 4 * XSLOT + 2 * ZSLOT, RED = DW_WAVES / 2 * TPW * 64 * 16 * 4;
    static constexpr int LDS = STAGE > RED ? STAGE : RED;
    static constexpr int XPER = (DW_RMAX * DW_ROWP * (CIN / 8) + 64 * DW_WAVES - 1) / (64 * DW_WAVES);
    static constexpr int ZPER = (DW_POS * (COUT / 8) + 64 * DW_WAVES - 1) / (64 * DW_WAVES);
};

#ifdef __HIP__
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
#else
typedef bf16x4 lds_bf16x4;
#endif
// 8 cells (rows a and b of this lane's two transposed reads) of one channel
__device__ __forceinline__ bf16x8 read_tr(char *a, char *b)
{
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4 *)a);
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4 *)b);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int CIN, int COUT>
__global__ void __launch_bounds__(64 * DW_WAVES) __attribute__((amdgpu_waves_per_eu(2, 2)))
dw_kernel(const DwGeom dg, const bf16 *__restrict__ X, const bf16 *__restrict__ dZ, float *__restrict__ partials)
{
    typedef DwCfg<CIN, COUT> C;
    constexpr int TPW = C::TPW, NC = CIN / 8, NZ = COUT / 8, NT = 64 * DW_WAVES;
    __shared__ __attribute__((aligned(16))) char lds[C::LDS];
    char *const xr = lds, *const zr = lds + 4 * C::XSLOT;
    const ConvGeom &g = dg.g;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tg = wave % C::TG, kg = wave / C::TG;
    // transposed reads: this lane's address is row kr (and kr + 4) of the 16
    // cells, 4 channels from ch; its result is column 16 * half + j
    const int half = (lane >> 4) & 1, j = lane & 15;
    const int kr = 8 * (lane >> 5) + (j >> 2);
    const int npos = dg.ry * dg.rz, nkb = (npos + 15) / 16;

    // the dZ slots past npos stay zero
    for (int e = tid * 16; e < 2 * C::ZSLOT; e += NT * 16) *reinterpret_cast<u32x4 *>(zr + e) = u32x4{0, 0, 0, 0};

    f32x16 acc[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.0f;

    u32x4 xv[C::XPER], zv[C::ZPER];
    int b = 0, y0 = 0, z0 = 0;
    auto load_x = [&](int xi) {
        const long long pb = ((long long)b * g.in[0] + xi) * g.in[1];
#pragma unroll
        for (int k = 0; k < C::XPER; ++k) {
            const int idx = k * NT + tid, cell = idx / NC, q = idx % NC;
            const int yi = y0 + cell / DW_ROWP, zi = z0 + cell % DW_ROWP;
            const bool in = cell / DW_ROWP < dg.ry + 2 && cell % DW_ROWP < dg.rz + 2 && xi < g.in[0] && yi < g.in[1] &&
                            zi < g.in[2];
            xv[k] = in ? *reinterpret_cast<const u32x4 *>(X + ((pb + yi) * g.in[2] + zi) * CIN + q * 8)
                       : u32x4{0, 0, 0, 0};
        }
    };
    auto store_x = [&](int xi) {
        char *slot = xr + (xi & 3) * C::XSLOT;
#pragma unroll
        for (int k = 0; k < C::XPER; ++k) {
            const int idx = k * NT + tid, cell = idx / NC, q = idx % NC;
            if (cell / DW_ROWP < dg.ry + 2 && cell % DW_ROWP < dg.rz + 2)
                *reinterpret_cast<u32x4 *>(slot + cell * C::XB + q * 16) = xv[k];
        }
    };
    auto load_z = [&](int x) {
        const long long pb = ((long long)b * g.out[0] + x) * g.out[1];
#pragma unroll
        for (int k = 0; k < C::ZPER; ++k) {
            const int idx = k * NT + tid, cell = idx / NZ, q = idx % NZ;
            const int r = cell * dg.magic >> 16, yi = y0 + r, zi = z0 + cell - r * dg.rz;
            const bool in = cell < npos && yi < g.out[1] && zi < g.out[2];
            zv[k] = in ? *reinterpret_cast<const u32x4 *>(dZ + ((pb + yi) * g.out[2] + zi) * COUT + q * 8)
                       : u32x4{0, 0, 0, 0};
        }
    };
    auto store_z = [&](int x) {
        char *slot = zr + (x & 1) * C::ZSLOT;
#pragma unroll
        for (int k = 0; k < C::ZPER; ++k) {
            const int idx = k * NT + tid;
            if (idx / NZ < npos) *reinterpret_cast<u32x4 *>(slot + idx * 16) = zv[k];
        }
    };

    for (long long item = blockIdx.x; item < dg.items; item += gridDim.x) {
        long long r = item;
        z0 = (int)(r % dg.nz) * dg.rz; r /= dg.nz;
        y0 = (int)(r % dg.ny) * dg.ry; r /= dg.ny;
        const int xs = (int)(r % dg.nxc) * dg.cx, xe = min(xs + dg.cx, g.out[0]);
        b = (int)(r / dg.nxc);
        __syncthreads();   // the zeroed dZ slots
#pragma unroll
        for (int k = 0; k < 3; ++k) { load_x(xs + k); store_x(xs + k); }
        load_z(xs);
        store_z(xs);
        __syncthreads();
        for (int x = xs; x < xe; ++x) {
            const bool more = x + 1 < xe;
            if (more) { load_x(x + 3); load_z(x + 1); }
            // this lane's part of the tiles' input addresses
            char *tb[TPW];
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                int tap, ch;
                if (CIN == 32) { tap = tg * TPW + t; ch = 16 * half + 4 * (j & 3); }
                else { tap = 4 * t + 2 * half + ((j & 3) >> 1); ch = 4 * (j & 1); }
                if (tap == 27) tap = 0;
                const int dx = tap / 9, dy = tap / 3 % 3, dz = tap % 3;
                tb[t] = xr + ((x + dx) & 3) * C::XSLOT + (dy * DW_ROWP + dz) * C::XB + ch * 2;
            }
            char *zb = zr + (x & 1) * C::ZSLOT + (COUT == 32 ? 16 * half : 0) * 2 + 8 * (j & 3);
            for (int kb = kg; kb < nkb; kb += C::KG) {
                const int i0 = kb * 16 + kr, i1 = i0 + 4;
                bf16x8 a = read_tr(zb + i0 * C::ZB, zb + i1 * C::ZB);
                if (COUT == 16 && half) a = zero8();
                const int c0 = i0 < npos ? i0 : npos - 1, c1 = i1 < npos ? i1 : npos - 1;
                const int r0 = c0 * dg.magic >> 16, r1 = c1 * dg.magic >> 16;
                const int o0 = (r0 * (DW_ROWP - dg.rz) + c0) * C::XB, o1 = (r1 * (DW_ROWP - dg.rz) + c1) * C::XB;
#pragma unroll
                for (int t = 0; t < TPW; ++t) {
                    bf16x8 bv = read_tr(tb[t] + o0, tb[t] + o1);
                    if (t == TPW - 1) {   // the bias columns
                        const bool one = CIN == 32 ? tg == C::TG - 1 : 2 * half + (j >> 3) == 3;
#pragma unroll
                        for (int i = 0; i < 8; ++i) bv[i] = one ? (bf16)1.0f : bv[i];
                    }
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bv, acc[t], 0, 0, 0);
                }
            }
            if (more) { store_x(x + 3); store_z(x + 1); }
            __syncthreads();
        }
    }

    // add the KG sums of every tile (halves, in a fixed order), then one
    // partial per workgroup: [column][32 couts]
    float *red = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int s = C::KG / 2; s >= 1; s >>= 1) {
        __syncthreads();
        if (kg >= s && kg < 2 * s) {
            float *o = red + ((kg - s) * C::TG + tg) * TPW * 1024 + lane * 4;
#pragma unroll
            for (int t = 0; t < TPW; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<f32x4 *>(o + t * 1024 + q * 256) =
                        f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
        }
        __syncthreads();
        if (kg < s) {
            const float *o = red + (kg * C::TG + tg) * TPW * 1024 + lane * 4;
#pragma unroll
            for (int t = 0; t < TPW; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(o + t * 1024 + q * 256);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[t][4 * q + i] += v[i];
                }
        }
    }
    if (kg == 0) {
        float *P = partials + (size_t)blockIdx.x * C::NTILES * 1024;
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4 *>(P + ((tg * TPW + t) * 32 + lane % 32) * 32 + 8 * q + 4 * (lane / 32)) =
                    f32x4{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
    }
}

// grad[tap][cin_real][cout_real] and, after it, the bias gradient: the sum
// over workgroups of the partials.  One block per (tap, cin), the last one for
// the bias column; 8 groups of 32 lanes (one per output channel) each sum
// every 8th workgroup in order, then the 8 group sums are added in order (a
// fixed order: deterministic).
__global__ void __launch_bounds__(256)
dw_reduce_kernel(const float *__restrict__ partials, int nwg, int cin_pad, int cin_real, int cout_real,
                 float *__restrict__ grad)
{
    __shared__ double red[8][32];
    const int tap = blockIdx.x / cin_real, ci = blockIdx.x % cin_real;   // tap 27: bias
    const int n = tap * cin_pad + ci;
    const int co = threadIdx.x & 31, grp = threadIdx.x >> 5;
    double s = 0.0;
#pragma unroll 8   // loads in flight: 10.4 -> 6.1 us for 256 partials of layer 2
    for (int w = grp; w < nwg; w += 8) s += (double)partials[((size_t)w * 28 * cin_pad + n) * 32 + co];
    red[grp][co] = s;
    __syncthreads();
    if (grp == 0 && co < cout_real) {
        double t = 0.0;
        for (int q = 0; q < 8; ++q) t += red[q][co];
        grad[(size_t)blockIdx.x * cout_real + co] = (float)t;
    }
}

// ---------------------------------------------------- weights, Adam --
// Parameter i of the network (W1, b1, W2, b2, W3, b3) to its places in the
// fragment-order bf16 weights: the forward layer's and (layers 2 and 3) the
// input-gradient convolution's (taps flipped, cin <-> cout); biases to their
// padded fp32 copies.  The padding stays as allocated, zero.
__device__ __forceinline__ void store_packed(const Packed &P, int i, float w)
{
    int layer = 0, cin = 5, cout = 32, base = 0;
    if (i >= 27 * 5 * 32 + 32) { layer = 1; cin = 32; base = 27 * 5 * 32 + 32; }
    if (i >= base + 27 * 32 * 32 + 32 && layer) { layer = 2; cout = 15; base += 27 * 32 * 32 + 32; }
    i -= base;
    if (i >= 27 * cin * cout) {
        P.bias[layer][i - 27 * cin * cout] = w;
        return;
    }
    // as a convolution of CIP (padded) input channels, COP outputs: input channel c, output n
    auto place = [&](int CIP, int tap, int c, int n) {
        const int tps = 32 / CIP, ks = (9 + tps - 1) / tps;
        const int dx = tap / 9, yz = tap % 9, s = yz / tps, k = yz % tps * CIP + c;
        return ((((n / 16) * ks + s) * 3 + dx) * 64 + k / 8 * 16 + n % 16) * 8 + k % 8;
    };
    const int n = i % cout, c = i / cout % cin, tap = i / (cout * cin);
    static_cast<bf16 *>(P.w[layer])[place(layer ? 32 : 8, tap, c, n)] = (bf16)w;
    if (layer) static_cast<bf16 *>(P.wt[layer])[place(layer == 1 ? 32 : 16, 26 - tap, n, c)] = (bf16)w;
}

__global__ void pack_kernel(const float *__restrict__ w, int n, const Packed P)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) store_packed(P, i, w[i]);
}

// Adam, and the updated parameters to their packed places: one launch where
// five packing kernels and three copies followed, 4 us each (Adam step of 8
// crops of 32^3: 399 -> 384 us).
__global__ void adam_kernel(float *__restrict__ w, const float *__restrict__ gr, float *__restrict__ m,
                            float *__restrict__ v, int n, float lr, float b1, float b2, float eps, float bc1,
                            float bc2, const Packed P)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float mh = mi / bc1, vh = vi / bc2;
    const float wi = w[i] - lr * mh / (sqrtf(vh) + eps);
    w[i] = wi;
    store_packed(P, i, wi);
}

// ----------------------------------------------- inputs, loss, update --
// Normalized primitives (bf16, 8 channels, 5 used) of a periodic n0 x n1 x n2
// SoA conserved state, for the box [o - halo, o - halo + dims) (wrapped),
// one box per batch item: boxes[b] = (sample, o0, o1, o2).
__global__ void __launch_bounds__(256)
prep_input_kernel(const PrepArgs a, const float *const *__restrict__ samples, const int *__restrict__ boxes,
                  bf16 *__restrict__ X, int *__restrict__ zero)
{
    if (zero && blockIdx.x == 0 && threadIdx.x == 0) *zero = 0;
    const long long per = (long long)a.dims[0] * a.dims[1] * a.dims[2];
    const long long total = per * a.B;
    const float V = a.ds * a.ds * a.ds, gm1 = a.gamma - 1.0f;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int b = (int)(e / per);
        long long r = e % per;
        const int z = (int)(r % a.dims[2]); r /= a.dims[2];
        const int y = (int)(r % a.dims[1]);
        const int x = (int)(r / a.dims[1]);
        const int *bx = boxes + 4 * b;
        const float *const *U = samples + 5 * bx[0];
        const int gx = ((bx[1] + x - a.halo) % a.n[0] + a.n[0]) % a.n[0];
        const int gy = ((bx[2] + y - a.halo) % a.n[1] + a.n[1]) % a.n[1];
        const int gz = ((bx[3] + z - a.halo) % a.n[2] + a.n[2]) % a.n[2];
        const long long c = ((long long)gx * a.n[1] + gy) * a.n[2] + gz;
        const float rho = U[0][c] / V;
        const float vx = U[1][c] / (rho * V), vy = U[2][c] / (rho * V), vz = U[3][c] / (rho * V);
        const float p = (U[4][c] / V - 0.5f * rho * (vx * vx + vy * vy + vz * vz)) * gm1;
        const float q[5] = {rho, vx, vy, vz, p};
        bf16x8 out = zero8();
#pragma unroll
        for (int f = 0; f < 5; ++f) {
            float v = (q[f] - a.shift[f]) * a.inv_scale[f];
            if (a.noise > 0.0f) {
                // counter-based normal variate (Box-Muller on two hashed uniforms)
                const uint32_t k = (uint32_t)(e * 5 + f);
                const uint32_t h1 = mix32(k ^ a.seed), h2 = mix32(k ^ (a.seed * 0x9E3779B9u + 0x7F4A7C15u));
                const float u1 = ((h1 >> 8) + 1u) * (1.0f / 16777217.0f), u2 = (h2 >> 8) * (1.0f / 16777216.0f);
                v += a.noise * sqrtf(-2.0f * logf(u1)) * cosf(6.2831853f * u2);
            }
            out[f] = (bf16)v;
        }
        *reinterpret_cast<bf16x8 *>(X + e * 8) = out;
    }
}

// Targets of a batch: R / out_scale over the loss box (wrapped), fp32 [B][L^3][5].
__global__ void __launch_bounds__(256)
prep_target_kernel(const PrepArgs a, const float *const *__restrict__ samples, const int *__restrict__ boxes,
                   float *__restrict__ T)
{
    const int L = a.dims[0];
    const long long per = (long long)L * L * L, total = per * a.B;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int b = (int)(e / per);
        long long r = e % per;
        const int z = (int)(r % L); r /= L;
        const int y = (int)(r % L);
        const int x = (int)(r / L);
        const int *bx = boxes + 4 * b;
        const float *const *R = samples + 5 * bx[0];
        const int gx = (bx[1] + x) % a.n[0], gy = (bx[2] + y) % a.n[1], gz = (bx[3] + z) % a.n[2];
        const long long c = ((long long)gx * a.n[1] + gy) * a.n[2] + gz;
#pragma unroll
        for (int f = 0; f < 5; ++f) T[e * 5 + f] = R[f][c] * a.inv_out[f];
    }
}

// Divergence loss over the L^3 box: P[c][q] = -sum_d (G[c+1][5d+q] - G[c+1-e_d][5d+q])
// (G on (L+1)^3, index c+1 = face c + e_d/2), loss = mean (P - T)^2 over cells and
// the 5 components; dG = dloss/dG (bf16, 16 channels, channel 15 zero); per-block
// partial loss sums.
// A face needs the errors of its cell and of three neighbours, each 15 loads
// over 64-byte cells (the cache's tag rate bounds them), so they are computed
// once: a workgroup takes a run of (y, z) positions of one batch item,
// flattened, and marches a few x planes with the last planes' errors (its
// positions and the Lg + 1 that follow them, the y and z neighbours) in LDS.
// 8 crops of 32^3: 20 us; four errors per thread from memory, 36 us.
constexpr int LOSS_THREADS = 512;
constexpr int LOSS_EXT = 960;   // positions with errors per run: L up to 830 (a box of which needs 300 GB)
struct LossGeom {
    int run, nrun;     // positions per run, runs per plane
    int cx, nxc;       // planes per item, items along x
    long long items;   // B * nrun * nxc
};
__global__ void __launch_bounds__(LOSS_THREADS)
loss_kernel(int L, const LossGeom lg, double N, const float *__restrict__ G, const float *__restrict__ T,
            bf16 *__restrict__ dG, double *__restrict__ loss_part)
{
    __shared__ float lds[3 * 5 * LOSS_EXT];
    __shared__ double red[LOSS_THREADS];
    const int Lg = L + 1, plane = Lg * Lg, ext = lg.run + Lg + 1, tid = threadIdx.x;
    const float scale = (float)(2.0 / N);
    double lsum = 0.0;
    for (long long item = blockIdx.x; item < lg.items; item += gridDim.x) {
        const int run = (int)(item % lg.nrun), xc = (int)(item / lg.nrun % lg.nxc);
        const long long b = item / lg.nrun / lg.nxc;
        const int p0 = run * lg.run, nown = min(lg.run, plane - p0), nerr = min(ext, plane - p0);
        const int xs = xc * lg.cx, xe = min(xs + lg.cx, Lg);
        // errors of the cells (cx, y - 1, z - 1) at positions p0 .. p0 + nerr - 1 (zero outside the box)
        auto errors = [&](int cx) {
            float *E = lds + (cx + 3) % 3 * 5 * ext;
            for (int i = tid; i < nerr; i += LOSS_THREADS) {
                const int gy = (p0 + i) / Lg, gz = (p0 + i) - gy * Lg;
                float e[5] = {0, 0, 0, 0, 0};
                if (cx >= 0 && cx < L && gy > 0 && gz > 0) {
                    const f32x4 *own = reinterpret_cast<const f32x4 *>(
                        G + ((b * Lg + cx + 1) * plane + p0 + i) * 16);
                    const f32x4 *xm = own - (long long)plane * 4, *ym = own - (long long)Lg * 4, *zm = own - 4;
                    const f32x4 a0 = own[0], a1 = own[1], a2 = own[2], a3 = own[3];
                    const f32x4 x0 = xm[0], x1 = xm[1], y1 = ym[1], y2 = ym[2], z2 = zm[2], z3 = zm[3];
                    const float gx0[5] = {a0[0], a0[1], a0[2], a0[3], a1[0]}, gx1[5] = {x0[0], x0[1], x0[2], x0[3], x1[0]};
                    const float gy0[5] = {a1[1], a1[2], a1[3], a2[0], a2[1]}, gy1[5] = {y1[1], y1[2], y1[3], y2[0], y2[1]};
                    const float gz0[5] = {a2[2], a2[3], a3[0], a3[1], a3[2]}, gz1[5] = {z2[2], z2[3], z3[0], z3[1], z3[2]};
                    const float *t = T + (((b * L + cx) * L + gy - 1) * L + gz - 1) * 5;
#pragma unroll
                    for (int q = 0; q < 5; ++q)
                        e[q] = -((gx0[q] - gx1[q]) + (gy0[q] - gy1[q]) + (gz0[q] - gz1[q])) - t[q];
                }
#pragma unroll
                for (int q = 0; q < 5; ++q) E[q * ext + i] = e[q];
            }
        };
        __syncthreads();   // the last item's reads are done
        errors(xs - 1);
        for (int gx = xs; gx < xe; ++gx) {
            errors(gx);
            __syncthreads();   // with three planes in LDS, the only one a plane needs
            const float *E0 = lds + (gx + 2) % 3 * 5 * ext, *E1 = lds + gx % 3 * 5 * ext;
            for (int i = tid; i < nown; i += LOSS_THREADS) {
                const int gy = (p0 + i) / Lg, gz = (p0 + i) - gy * Lg;
                bf16x8 lo = zero8(), hi = zero8();
#pragma unroll
                for (int q = 0; q < 5; ++q) {
                    const float e0 = E0[q * ext + i];
                    lsum += (double)e0 * e0;   // (zero where there is no cell)
                    // d/dG[g][5d+q]: -e(c) from cell c = g-1, + e(c + e_d) from cell g-1+e_d
                    const float n[3] = {E1[q * ext + i], gy < L ? E0[q * ext + i + Lg] : 0.0f,
                                        gz < L ? E0[q * ext + i + 1] : 0.0f};
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const int ch = 5 * d + q;
                        const bf16 v = (bf16)(scale * (-e0 + n[d]));
                        if (ch < 8) lo[ch] = v;
                        else hi[ch - 8] = v;
                    }
                }
                bf16 *out = dG + ((b * Lg + gx) * plane + p0 + i) * 16;
                *reinterpret_cast<bf16x8 *>(out) = lo;
                *reinterpret_cast<bf16x8 *>(out + 8) = hi;
            }
        }
    }
    red[tid] = lsum;
    __syncthreads();
    for (int s = LOSS_THREADS / 2; s > 0; s >>= 1) {
        if (tid < s) red[tid] += red[tid + s];
        __syncthreads();
    }
    if (tid == 0) loss_part[blockIdx.x] = red[0] / N;
}

// Host-array staging: fp32 [cells][creal] -> bf16 [cells][cpad]
__global__ void to_bf16_kernel(const float *__restrict__ x, long long ncells, int creal, int cpad, bf16 *__restrict__ y)
{
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ncells * cpad) return;
    const long long m = e / cpad;
    const int c = (int)(e % cpad);
    y[e] = (bf16)(c < creal ? x[m * creal + c] : 0.0f);
}

// ------------------------------------------------------------ launches --
static ConvGeom geom(int B, const int in[3], int pad)
{
    ConvGeom g;
    g.B = B;
    for (int d = 0; d < 3; ++d) {
        g.in[d] = in[d];
        g.out[d] = pad ? in[d] + 2 : in[d] - 2;
    }
    g.ncells = (long long)B * g.out[0] * g.out[1] * g.out[2];
    return g;
}

static int grid_for(long long n, long long per, int cap)
{
    long long b = (n + per - 1) / per;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (int)b;
}

static int cu_count()
{
    static int n = 0;
    if (!n) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            n = v;
        else
            n = 256;
    }
    return n;
}

// Rectangles of at most RING_POS positions with rz + 2 <= RING_ROWP and
// ry + 2 <= RING_RMAX: those with the least work per plane (a workgroup computes
// RING_POS positions whatever it owns, and stages the halo); x chunks: the
// shortest schedule on the CUs, an item costing its planes plus 3.
static RingGeom ring_geom(const ConvGeom &g)
{
    RingGeom r;
    r.g = g;
    const int o0 = g.out[0], o1 = g.out[1], o2 = g.out[2];
    long long best = -1;
    const int nz0 = (o2 + RING_ROWP - 3) / (RING_ROWP - 2);
    for (int nz = nz0; nz <= nz0 + 4 && nz <= o2; ++nz) {
        const int rz = (o2 + nz - 1) / nz;
        int ry = RING_POS / rz;
        if (ry > RING_RMAX - 2) ry = RING_RMAX - 2;
        if (ry > o1) ry = o1;
        const int ny = (o1 + ry - 1) / ry;
        ry = (o1 + ny - 1) / ny;
        const long long cost = (long long)ny * nz * (4 * RING_POS + (ry + 2) * (rz + 2));
        if (best < 0 || cost < best) {
            best = cost;
            r.ry = ry; r.rz = rz;
            r.ny = ny; r.nz = (o2 + rz - 1) / rz;
        }
    }
    const long long cols = (long long)g.B * r.ny * r.nz, cus = cu_count();
    best = -1;
    r.cx = o0;
    for (int cx = o0; cx >= 1; --cx) {
        const long long rounds = (cols * ((o0 + cx - 1) / cx) + cus - 1) / cus, cost = rounds * (cx + 3);
        if (best < 0 || cost < best) { best = cost; r.cx = cx; }
    }
    r.nxc = (o0 + r.cx - 1) / r.cx;
    r.items = cols * r.nxc;
    return r;
}

int conv(int layer, int mode, int B, const int in[3], const void *X, const void *Wp, const float *bias, float *Z,
         void *Xout, float *Y, const float *Zprev, hipStream_t s)
{
    const int pad = mode == CONV_BWD ? 2 : 0;
    const ConvGeom g = geom(B, in, pad);
    for (int d = 0; d < 3; ++d)
        if (g.out[d] < 1) return -1;
    const RingGeom rg = ring_geom(g);
    const bf16 *x = static_cast<const bf16 *>(X);
    const bf16x8 *w = static_cast<const bf16x8 *>(Wp);
    bf16 *xo = static_cast<bf16 *>(Xout);
#define DG_CONV(CI, CO, E, P)                                                                                    \
    do {                                                                                                         \
        const long long fit = (long long)cu_count() * (4 * ConvCfg<CI, CO>::EU / ConvCfg<CI, CO>::WAVES);         \
        hipLaunchKernelGGL((conv_ring_kernel<CI, CO, E, P>), dim3((unsigned)(rg.items < fit ? rg.items : fit)),  \
                           dim3(ConvCfg<CI, CO>::THREADS), 0, s, rg, x, w, bias, Z, xo, Y, Zprev);               \
    } while (0)
    if (layer == 1) {
        if (mode == CONV_TRAIN) DG_CONV(8, 32, EPI_TRAIN, 0);
        else if (mode == CONV_INFER) DG_CONV(8, 32, EPI_INFER, 0);
        else return -1;
    } else if (layer == 2) {
        if (mode == CONV_TRAIN) DG_CONV(32, 32, EPI_TRAIN, 0);
        else if (mode == CONV_INFER) DG_CONV(32, 32, EPI_INFER, 0);
        else DG_CONV(32, 32, EPI_BWD, 2);   // input gradient of layer 2 (dZ2 -> dZ1)
    } else if (layer == 3) {
        if (mode == CONV_BWD) DG_CONV(16, 32, EPI_BWD, 2);   // input gradient of layer 3 (dG -> dZ2)
        else if (mode == CONV_OUT16) DG_CONV(32, 16, EPI_OUT16, 0);
        else DG_CONV(32, 16, EPI_OUT, 0);
    } else {
        return -1;
    }
#undef DG_CONV
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Rectangles of at most 7 x 46 outputs: rz balanced over the extent, ry the
// one that leaves the fewest 16-cell blocks (rounded up to the waves that
// split them); x chunks so that the work items fill nwg workgroups once.
static DwGeom dw_geom(const ConvGeom &g, int kgroups, int nwg)
{
    DwGeom d;
    d.g = g;
    d.nz = (g.out[2] + DW_ROWP - 3) / (DW_ROWP - 2);
    d.rz = (g.out[2] + d.nz - 1) / d.nz;
    d.magic = (65536 + d.rz - 1) / d.rz;
    long long best = -1;
    d.ry = 1;
    for (int ry = 1; ry <= DW_RMAX - 2 && ry <= g.out[1]; ++ry) {
        const long long rows = (g.out[1] + ry - 1) / ry, blocks = (ry * d.rz + 16 * kgroups - 1) / (16 * kgroups);
        const long long cost = rows * (4 * blocks + ry + 4);   // MFMAs, staging and a barrier per plane
        if (best < 0 || cost <= best) { best = cost; d.ry = ry; }
    }
    d.ny = (g.out[1] + d.ry - 1) / d.ry;
    const long long cols = (long long)g.B * d.ny * d.nz;
    long long nxc = nwg / cols;
    if (nxc > g.out[0]) nxc = g.out[0];
    if (nxc < 1) nxc = 1;
    d.cx = (int)((g.out[0] + nxc - 1) / nxc);
    d.nxc = (g.out[0] + d.cx - 1) / d.cx;
    d.items = cols * d.nxc;
    return d;
}

template <int CIN, int COUT>
static int launch_dw(const ConvGeom &g, const void *X, const void *dZ, float *partials, int nwg, hipStream_t s)
{
    const DwGeom d = dw_geom(g, DwCfg<CIN, COUT>::KG, nwg);
    const int blocks = (int)(d.items < nwg ? d.items : nwg);
    hipLaunchKernelGGL((dw_kernel<CIN, COUT>), dim3(blocks), dim3(64 * DW_WAVES), 0, s, d, static_cast<const bf16 *>(X),
                       static_cast<const bf16 *>(dZ), partials);
    return blocks;
}

int dw(int layer, int B, const int in[3], const void *X, const void *dZ, float *partials, int nwg, float *grad,
       hipStream_t s)
{
    const ConvGeom g = geom(B, in, 0);
    const int cin_pad = layer == 1 ? 8 : 32, cin_real = layer == 1 ? 5 : 32, cout_real = layer == 3 ? 15 : 32;
    const int blocks = layer == 1 ? launch_dw<8, 32>(g, X, dZ, partials, nwg, s)
                       : layer == 2 ? launch_dw<32, 32>(g, X, dZ, partials, nwg, s)
                                    : launch_dw<32, 16>(g, X, dZ, partials, nwg, s);
    hipLaunchKernelGGL(dw_reduce_kernel, dim3(27 * cin_real + 1), dim3(256), 0, s, partials, blocks, cin_pad, cin_real,
                       cout_real, grad);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int pack(const float *w, int n, const Packed &P, hipStream_t s)
{
    hipLaunchKernelGGL(pack_kernel, dim3((n + 255) / 256), dim3(256), 0, s, w, n, P);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int pack_elems(int layer, int transpose)
{
    const int cin_pad = layer == 1 ? 8 : 32, cout_pad = layer == 3 ? 16 : 32;
    const int CIP = transpose ? cout_pad : cin_pad, COP = transpose ? cin_pad : cout_pad;
    const int tps = 32 / CIP, ks = (9 + tps - 1) / tps;
    return COP / 16 * ks * 3 * 64 * 8;
}

int adam(float *w, const float *g, float *m, float *v, int n, float lr, float b1, float b2, float eps, long long t,
         const Packed &P, hipStream_t s)
{
    const float bc1 = 1.0f - powf(b1, (float)t), bc2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(adam_kernel, dim3((n + 255) / 256), dim3(256), 0, s, w, g, m, v, n, lr, b1, b2, eps, bc1, bc2,
                       P);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int prep_input(const PrepArgs &a, const float *const *samples, const int *boxes, void *X, hipStream_t s, int *zero)
{
    const long long n = (long long)a.B * a.dims[0] * a.dims[1] * a.dims[2];
    hipLaunchKernelGGL(prep_input_kernel, dim3(grid_for(n, 256, 16384)), dim3(256), 0, s, a, samples, boxes,
                       static_cast<bf16 *>(X), zero);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int prep_target(const PrepArgs &a, const float *const *samples, const int *boxes, float *T, hipStream_t s)
{
    const long long n = (long long)a.B * a.dims[0] * a.dims[0] * a.dims[0];
    hipLaunchKernelGGL(prep_target_kernel, dim3(grid_for(n, 256, 16384)), dim3(256), 0, s, a, samples, boxes, T);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Runs of equal length whose errors one pass of the workgroup computes (longer
// ones where a row alone is more), and items for the nblk workgroups.
int loss(int B, int L, const float *G, const float *T, void *dG, double *loss_part, int nblk, hipStream_t s)
{
    const int Lg = L + 1, plane = Lg * Lg;
    LossGeom lg;
    const int fit = LOSS_THREADS - Lg - 1 > LOSS_THREADS / 4 ? LOSS_THREADS - Lg - 1 : LOSS_THREADS / 4;
    lg.nrun = (plane + fit - 1) / fit;
    lg.run = (plane + lg.nrun - 1) / lg.nrun;
    const long long cols = (long long)B * lg.nrun;
    long long nxc = (nblk + cols - 1) / cols;
    if (nxc > Lg) nxc = Lg;
    lg.cx = (int)((Lg + nxc - 1) / nxc);
    lg.nxc = (Lg + lg.cx - 1) / lg.cx;
    lg.items = cols * lg.nxc;
    if (lg.run + Lg + 1 > LOSS_EXT) return -1;
    hipLaunchKernelGGL(loss_kernel, dim3(nblk), dim3(LOSS_THREADS), 0, s, L, lg, (double)B * L * L * L * 5, G, T,
                       static_cast<bf16 *>(dG), loss_part);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int to_bf16(const float *x, long long ncells, int creal, int cpad, void *y, hipStream_t s)
{
    const long long n = ncells * cpad;
    hipLaunchKernelGGL(to_bf16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, ncells, creal, cpad,
                       static_cast<bf16 *>(y));
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace cnn
}  // namespace dg
