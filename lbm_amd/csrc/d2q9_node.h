// d2q9_node.h -- one lattice node: parameter block, storage forms, pulls,
// obstacle links, walls, moments and collision.  Shared by the one-iteration
// kernels (d2q9_fused.hip) and the multi-iteration ones (d2q9_tile.hip).
#pragma once
#include "d2q9_common.h"
#include "d2q9_zouhe.h"
#include "../../include/lbm_d2q9.h"

namespace lbm {

// ------------------------------------------------------------------ links --
// One obstacle link (fluid node `cell`, direction q towards the solid), with
// the reads of its bounce-back value resolved to (plane, node) pairs and the
// interpolation factors of nb.py:97-104 formed on the host in double.
struct LinkRec {
    int32_t cell;          // fluid node, x*ny + y
    int32_t cellB, cellC;  // nodes of the 2nd and 3rd reads
    int8_t q, qb, planeB, planeC;
    int32_t mode;          // 0 plain bounce-back, 1 interpolated
    int32_t dslot;         // position of the link in plan order (drag row)
    double c0, c1, c2;     // value = (c0*A + c1*B) + c2*C
};

struct Params {
    const void *src;       // post-collision field of iteration it-1 (storage form)
    void *dst;             // post-collision field of iteration it
    const double *g0;      // INIT: populations of iteration 0, double[9][N]
    double *g_out;         // EPILOGUE: post-boundary populations, double[9][N]
    double *gup_out;       // EPILOGUE: src converted to double[9][N]
    double *rho_out, *u_out;
    int nx, ny, N;
    uint32_t magic;        // floor(2^32 / ny) + 1, for node -> (x, y)
    double om_p, om_m, b0, a1, a2, a3, a4;
    float omf_p, omf_m;    // om_p and om_m rounded to float (the float forms' rates)
    int bc_bottom, bc_left, bc_top, bc_right, corners;
    const double *pool;    // inlet side arrays
    const int *inlet_off;  // [ring][5] offsets into pool
    const double *amp;     // separable inlets: amp[row * amp_stride + side] (or null)
    int amp_stride;
    const double *prof[5]; // separable inlets: per-side profiles
    int ring;
    const int *base;       // device int: row of iteration (it0-1) in graph replays
    int k;                 // row = (*base + k) mod ring  -- row of iteration it-1
    const int *tile_slot;  // [n_tiles] -1 or slot of the tile's link offsets
    const int *cell_off;   // [n_slots][tile_cells+1]
    const uint32_t *cell_mask; // [n_slots][tile_cells/32] bit set = node has links
    const int *wave_rng;   // float forms: [n_tiles][rng_stride] link-record bounds of
    int rng_stride;        // the tile's 64-node runs (every tile; equal bounds: no links)
    const uint32_t *run_bits; // float forms: bit r set = 64-node run r (node >> 6) has links
    int n_main;            // work-groups of interior tiles (the rest do the perimeter)
    int n_perim;           // perimeter nodes
    const LinkRec *links;  // sorted by node
    double *drag_ring;     // [ring][n_links]
    int n_links;
    const int *link_cells; // DRAG: distinct link nodes
    int n_link_cells;
    int tile_shift;        // log2(tile_cells)
    int rev;               // sweep the tiles last first (odd iterations, large lattices)
    int blk_shift;         // log2 of the tiles per XCD block (0: dispatch order)
    // Q16: h_q = qo[q] + qs[q] * i (decode); i = rint(h_q * qi[q] + qc[q]),
    // clamped to [-32767, 32767] (encode); qi = 1/qs, qc = -qo/qs.  qtab holds
    // the same four rows in device memory for directions known only at run
    // time (obstacle links): indexing these arrays with a run-time value would
    // move the whole parameter block to scratch memory.
    float qs[9], qo[9], qi[9], qc[9];
    const float *qtab;     // [4][9]: qs, qo, qi, qc
};

// ---------------------------------------------------------------- storage --
// A state buffer holds nine population planes of N nodes (plane q, node
// x*ny + y).  ld(p, buf, q, node) returns the population f_q; the float forms
// store a deviation and ldh returns h_q = f_q - w_q; sth stores h_q.
//   F64             f_q in double
//   F32, F16, BF16  h_q in float, IEEE half or bfloat16
//   F16E            g_q = h_q - E_q(v) in IEEE half, with
//                   E_q(v) = w_q (3 c_q.v + 4.5 (c_q.v)^2 - 1.5 v.v)
//                   the equilibrium deviation at the node's velocity v rounded
//                   to half precision; a tenth plane holds v as packed (vx, vy)
//                   half pairs.  g_q is the density and non-equilibrium part
//                   of h_q (~1e-3 against ~2e-2 for h_q in a u ~ 0.05 flow), so
//                   half precision resolves it 10-30 times finer.  Writer and
//                   reader evaluate E_q from the same half-precision v with the
//                   same operations, so the shift cancels exactly.
//   Q16             h_q in 16-bit fixed point on a per-direction affine map,
//                   h_q = qo[q] + qs[q] i with i in [-32767, 32767]: the 65535
//                   levels cover the range of h_q the flow can reach (set by
//                   the caller from its velocity bound), uniformly, where IEEE
//                   half spends most of its codes near zero.  Values outside
//                   the range are clamped to it.
template <int S> struct Store;

__host__ __device__ constexpr bool is16(int S)
{
    return S == LBM_STORE_F16 || S == LBM_STORE_BF16 || S == LBM_STORE_F16E ||
           S == LBM_STORE_Q16 || S == LBM_STORE_F16E8;
}

// Float -> half conversions are written as the instruction itself, so the
// compiler cannot fold the preceding multiply-add into a mixed-precision FMA
// that rounds to half once (v_fma_mixlo_f16): every kernel then rounds twice,
// to float and to half, and all kernel shapes store identical values.  (An
// empty asm on the operand did the same with a register move a value.)
__device__ __forceinline__ _Float16 to_half(float v)
{
    uint32_t h;
    asm("v_cvt_f16_f32 %0, %1" : "=v"(h) : "v"(v));
    return __builtin_bit_cast(_Float16, (uint16_t)h);
}
// two of them in one instruction, a in the low half (each rounds as to_half)
__device__ __forceinline__ uint32_t to_half2(float a, float b)
{
    uint32_t h;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(h) : "v"(a), "v"(b));
    return h;
}
// the low half of w (as an instruction: a conversion the compiler knows moves
// up to the load it waits for)
__device__ __forceinline__ float from_half(uint32_t w)
{
    float r;
    asm("v_cvt_f32_f16 %0, %1" : "=v"(r) : "v"(w));
    return r;
}
// e + the low / high half of w: one exact product by 1, one rounding
__device__ __forceinline__ float add_lo(float e, uint32_t w)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(e));
    return r;
}
__device__ __forceinline__ float add_hi(float e, uint32_t w)
{
    float r;
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(e));
    return r;
}

// F16E: offset (in halves) of the velocity plane, 256-byte aligned
__host__ __device__ constexpr size_t vel_offset(int N) { return ((size_t)9 * N + 127) / 128 * 128; }

// 16-bit forms: a plane element through a base pointer that is uniform over
// the work-group (kept in scalar registers) and a 32-bit byte offset shared
// by all planes of a node, so that each access is one global load or store
// with a scalar base and no 64-bit address arithmetic per plane (offsets of
// 2-byte elements stay below 2^32 for any int node count).
template <class E>
__device__ __forceinline__ E ld_off(const void *base, uint32_t off)
{
    return *reinterpret_cast<const E *>(static_cast<const char *>(base) + off);
}
template <class E>
__device__ __forceinline__ void st_off(void *base, uint32_t off, E v)
{
    using gchar = __attribute__((address_space(1))) char;
    using gE = __attribute__((address_space(1))) E;
    *(gE *)((gchar *)base + off) = v;
}
// ld_off of a base that has been through sbase (a plain load of it is a flat one)
template <class E>
__device__ __forceinline__ E ld_base(const void *base, uint32_t off)
{
    using gchar = __attribute__((address_space(1))) const char;
    using gE = __attribute__((address_space(1))) const E;
    return *(gE *)((gchar *)base + off);
}
// A uniform pointer through readfirstlane: the compiler keeps each plane's
// base in scalar registers instead of deriving one plane's address from the
// previous one with per-lane 64-bit additions.
template <class T>
__device__ __forceinline__ T *sbase(T *ptr)
{
    const uint64_t v = reinterpret_cast<uint64_t>(ptr);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<T *>(((uint64_t)hi << 32) | lo);
}

template <> struct Store<LBM_STORE_F64> {
    using s_t = double;
    using T = double;
    static __device__ __forceinline__ T ld(const Params &p, const s_t *b, int q, size_t c)
    {
        return b[(size_t)q * p.N + c];
    }
    static __device__ __forceinline__ void st(const Params &, s_t *b, int, size_t i, T v)
    {
        b[i] = v;
    }
};

template <> struct Store<LBM_STORE_F32> {
    using s_t = float;
    using T = float;
    static __device__ __forceinline__ float ldh(const Params &p, const s_t *b, int q, size_t c)
    {
        return b[(size_t)q * p.N + c];
    }
    static __device__ __forceinline__ void sth(const Params &, s_t *b, int, size_t i, float h)
    {
        b[i] = h;
    }
    static __device__ __forceinline__ T ld(const Params &p, const s_t *b, int q, size_t c)
    {
        return weight<float>(q) + ldh(p, b, q, c);
    }
};

template <> struct Store<LBM_STORE_F16> {
    using s_t = _Float16;
    using T = float;
    static __device__ __forceinline__ float dec(const Params &, int, s_t raw) { return (float)raw; }
    static __device__ __forceinline__ s_t enc(const Params &, int, float h) { return to_half(h); }
    static __device__ __forceinline__ float ldh(const Params &p, const s_t *b, int q, size_t c)
    {
        return (float)b[(size_t)q * p.N + c];
    }
    static __device__ __forceinline__ void sth(const Params &, s_t *b, int, size_t i, float h)
    {
        b[i] = to_half(h);
    }
    static __device__ __forceinline__ T ld(const Params &p, const s_t *b, int q, size_t c)
    {
        return weight<float>(q) + ldh(p, b, q, c);
    }
};

__device__ __forceinline__ uint16_t f32_to_bf16(float v)
{
    uint32_t u = __float_as_uint(v);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
    return (uint16_t)(u >> 16);
}

template <> struct Store<LBM_STORE_BF16> {
    using s_t = uint16_t;
    using T = float;
    static __device__ __forceinline__ float dec(const Params &, int, s_t raw)
    {
        return __uint_as_float((uint32_t)raw << 16);
    }
    static __device__ __forceinline__ s_t enc(const Params &, int, float h) { return f32_to_bf16(h); }
    static __device__ __forceinline__ float ldh(const Params &p, const s_t *b, int q, size_t c)
    {
        return __uint_as_float((uint32_t)b[(size_t)q * p.N + c] << 16);
    }
    static __device__ __forceinline__ void sth(const Params &, s_t *b, int, size_t i, float h)
    {
        b[i] = f32_to_bf16(h);
    }
    static __device__ __forceinline__ T ld(const Params &p, const s_t *b, int q, size_t c)
    {
        return weight<float>(q) + ldh(p, b, q, c);
    }
};

// Q16 encode: x = h qi + qc with qc = 1.5 * 2^23 - m (one FMA): the sum lies
// in [2^23, 2^24), where floats are the integers, so x is rounded to
// 1.5 * 2^23 + rint(h / qs) - m, whose low 16 bits are the code i in two's
// complement; x is clamped to the codes -32767 .. 32767.  A non-finite h
// gets the code -32768, which the density sum turns back into a NaN.  The
// multiply-add goes through an empty asm so that every kernel shape rounds
// it the same way.
constexpr float Q16_MAGIC = 12582912.0f;   // 1.5 * 2^23
__device__ __forceinline__ uint16_t q16_encode(float h, float qi, float qc)
{
    float x = __builtin_fmaf(h, qi, qc);
    asm("" : "+v"(x));
    const float c = __builtin_fminf(__builtin_fmaxf(x, Q16_MAGIC - 32767.0f), Q16_MAGIC + 32767.0f);
    return x == x ? (uint16_t)(__float_as_uint(c) & 0xffffu) : (uint16_t)0x8000u;
}

__device__ __forceinline__ float q16_decode(int16_t i, float qs, float qo)
{
    return __builtin_fmaf(qs, (float)i, qo);
}

// Affine-map coefficient `row` (0 qs, 1 qo, 2 qi, 3 qc) of direction q: from
// the kernel arguments when q is a compile-time constant after inlining (the
// unrolled node loops), else from the device table.
__device__ __forceinline__ float q16_coef(const Params &p, int row, int q)
{
    if (__builtin_constant_p(q)) {
        const float *r = row == 0 ? p.qs : row == 1 ? p.qo : row == 2 ? p.qi : p.qc;
        return r[q];
    }
    return p.qtab[row * 9 + q];
}

template <> struct Store<LBM_STORE_Q16> {
    using s_t = int16_t;
    using T = float;
    static __device__ __forceinline__ float dec(const Params &p, int q, s_t raw)
    {
        return q16_decode(raw, q16_coef(p, 0, q), q16_coef(p, 1, q));
    }
    static __device__ __forceinline__ s_t enc(const Params &p, int q, float h)
    {
        return (int16_t)q16_encode(h, q16_coef(p, 2, q), q16_coef(p, 3, q));
    }
    static __device__ __forceinline__ float ldh(const Params &p, const s_t *b, int q, size_t c)
    {
        return q16_decode(b[(size_t)q * p.N + c], q16_coef(p, 0, q), q16_coef(p, 1, q));
    }
    static __device__ __forceinline__ void sth(const Params &p, s_t *b, int q, size_t i, float h)
    {
        b[i] = (int16_t)q16_encode(h, q16_coef(p, 2, q), q16_coef(p, 3, q));
    }
    static __device__ __forceinline__ T ld(const Params &p, const s_t *b, int q, size_t c)
    {
        return weight<float>(q) + ldh(p, b, q, c);
    }
};

// F16E: E_q(v), explicit fmaf only, so every caller rounds identically
// c_q.v is taken as +-vx, +-vy or their sum (no multiplications by the
// integer components, which the compiler may not drop without fast-math), and
// E_q = cu (3 w_q + 4.5 w_q cu) - 1.5 w_q v.v with the products of the weights
// folded into constants (three operations after v.v and cu); q may be a
// run-time value (the link path), the selection then yields the same
// operations.  Writer and reader evaluate it on the same half-precision
// velocity, so the shift cancels exactly whatever its own rounding.
__device__ __forceinline__ float eq_shift(int q, float vx, float vy)
{
    const float vv = __builtin_fmaf(vy, vy, vx * vx);
    const float ax = CX[q] > 0 ? vx : -vx, ay = CY[q] > 0 ? vy : -vy;
    const float cu = CY[q] == 0 ? (CX[q] == 0 ? 0.0f : ax) : (CX[q] == 0 ? ay : ax + ay);
    const float w = weight<float>(q);
    return __builtin_fmaf(cu, __builtin_fmaf(4.5f * w, cu, 3.0f * w), (-1.5f * w) * vv);
}

// The velocity word of the shifted forms.  F16E: (vx, vy) as IEEE halves in
// 32 bits.  F16E8: (vx, vy) as 8-bit fixed point in 16 bits, steps of 2^-9,
// |v| <= 127/512 (clamped; the lattice speed of sound is 0.577 and the flows
// stay far below 0.25): the shift then differs from the node's exact
// equilibrium deviation by at most 3 w_q |c_q| 2^-10 more than with halves,
// still well under the stored residual, for 2 bytes less per node each way.
template <int S> struct Vel;
template <> struct Vel<LBM_STORE_F16E> {
    using w_t = uint32_t;
    static __device__ __forceinline__ w_t pack(float ux, float uy)
    {
        const _Float16 hx = to_half(ux), hy = to_half(uy);
        return (uint32_t)__builtin_bit_cast(uint16_t, hx) |
               ((uint32_t)__builtin_bit_cast(uint16_t, hy) << 16);
    }
    static __device__ __forceinline__ void unpack(w_t v, float &vx, float &vy)
    {
        vx = (float)__builtin_bit_cast(_Float16, (uint16_t)(v & 0xffffu));
        vy = (float)__builtin_bit_cast(_Float16, (uint16_t)(v >> 16));
    }
};
template <> struct Vel<LBM_STORE_F16E8> {
    using w_t = uint16_t;
};

// F16E8 velocity word: a = rint(512 vx), b = rint(512 vy), clamped to
// -127..127, as two's-complement bytes (a low).  Rounding by the magic number
// 1.5 * 2^23 (one FMA, round to nearest even, the integer in the low bits of
// the sum) and a median clamp; a and b come back as integer-valued floats.
__device__ __forceinline__ uint16_t e8_pack(float ux, float uy, float &a, float &b)
{
    constexpr float M = 12582912.0f;   // 1.5 * 2^23
    const float xa = __builtin_amdgcn_fmed3f(__builtin_fmaf(ux, 512.0f, M), M - 127.0f, M + 127.0f);
    const float xb = __builtin_amdgcn_fmed3f(__builtin_fmaf(uy, 512.0f, M), M - 127.0f, M + 127.0f);
    a = xa - M;
    b = xb - M;
    return (uint16_t)((__float_as_uint(xa) & 0xffu) | ((__float_as_uint(xb) & 0xffu) << 8));
}

// the two signed bytes of the word as floats (one byte-select convert each)
__device__ __forceinline__ void e8_unpack(uint32_t w, float &a, float &b)
{
    a = (float)((int32_t)(w << 24) >> 24);
    b = (float)((int32_t)(w << 16) >> 24);
}

// E_q of F16E8 on the integers (a, b) = 512 v: with cu = c_q.(a, b) and
// pv = c_q x (a, b) (the component across c_q), v.v = (cu^2 + pv^2) / |c_q|^2
// / 512^2 and
//   E_q = w_q (3 c.v + 4.5 (c.v)^2 - 1.5 v.v) = cu (K2 + K1 cu) - K3 pv^2,
//   E_0 = -K0 (a^2 + b^2),
// K2 = 3 w / 512, K1 = (4.5 - 1.5 / |c|^2) w / 512^2, K3 = 1.5 w / |c|^2 / 512^2.
// cu and pv are small integers (exact in float); the signs of c fold into
// the operands.  q may be a run-time value (the link path) and then yields
// the same operations on the same constants.
__host__ __device__ constexpr double e8_w(int q) { return q == 0 ? 4.0 / 9.0 : (q <= 4 ? 1.0 / 9.0 : 1.0 / 36.0); }
__host__ __device__ constexpr double e8_c2(int q) { return q <= 4 ? 1.0 : 2.0; }
__device__ __forceinline__ float e8_k0() { return (float)(1.5 * e8_w(0) / 262144.0); }
__device__ __forceinline__ float e8_k1(int q) { return (float)((4.5 - 1.5 / e8_c2(q)) * e8_w(q) / 262144.0); }
__device__ __forceinline__ float e8_k2(int q) { return (float)(3.0 * e8_w(q) / 512.0); }
__device__ __forceinline__ float e8_k3(int q) { return (float)(1.5 / e8_c2(q) * e8_w(q) / 262144.0); }
__device__ __forceinline__ float e8_cu(int q, float a, float b)
{
    const float ax = CX[q] > 0 ? a : -a, by = CY[q] > 0 ? b : -b;
    return CY[q] == 0 ? ax : (CX[q] == 0 ? by : ax + by);
}
__device__ __forceinline__ float e8_pv(int q, float a, float b)
{
    // c x v = cx b - cy a
    const float bx = CX[q] > 0 ? b : -b, ay = CY[q] > 0 ? -a : a;
    return CY[q] == 0 ? bx : (CX[q] == 0 ? ay : bx + ay);
}
// E_q itself: the writer stores half(h - E_q), the reader adds the same E_q
// back, so the shift cancels exactly whatever its own rounding (a reader that
// folded the residual into the multiply-add chain would differ from the
// writer by a float rounding of E, a bias the 200 000-iteration Turek run
// shows: max-Cl error 9.8e-4 against 5.9e-4)
__device__ __forceinline__ float e8_shift(int q, float a, float b)
{
    if (q == 0) {
        const float k = -e8_k0();
        return __builtin_fmaf(a * k, a, (b * k) * b);
    }
    const float cu = e8_cu(q, a, b), pv = e8_pv(q, a, b);
    const float t = __builtin_fmaf(e8_k1(q), cu, e8_k2(q));
    return __builtin_fmaf(cu, t, (pv * -e8_k3(q)) * pv);
}
// the nine of a node: an opposite pair shares the term in pv and, up to its
// sign, cu (the values of e8_shift)
__device__ __forceinline__ void e8_shifts(float a, float b, float *e)
{
    e[0] = e8_shift(0, a, b);
#pragma unroll
    for (int q = 1; q < 9; q += 2) {
        const float cu = e8_cu(q, a, b), pv = e8_pv(q, a, b), P = (pv * -e8_k3(q)) * pv;
        e[q] = __builtin_fmaf(cu, __builtin_fmaf(cu, e8_k1(q), e8_k2(q)), P);
        e[q + 1] = __builtin_fmaf(-cu, __builtin_fmaf(cu, -e8_k1(q), e8_k2(q)), P);
    }
}
__device__ __forceinline__ float e8_dec(int q, float a, float b, float r)
{
    float e = e8_shift(q, a, b);
    asm("" : "+v"(e));   // E_q as the writer rounds it, not fused with r
    return e + r;
}

// F16E / F16E8: g_q = h_q - E_q(v) in IEEE half with the velocity word in a
// tenth plane (256-byte aligned)
template <int S> struct StoreShifted {
    using s_t = _Float16;
    using T = float;
    using w_t = typename Vel<S>::w_t;
    static __device__ __forceinline__ const w_t *vel(const s_t *b, int N)
    {
        return reinterpret_cast<const w_t *>(b + vel_offset(N));
    }
    static __device__ __forceinline__ float dec(int q, s_t raw, w_t v)
    {
        if constexpr (S == LBM_STORE_F16E8) {
            float a, b;
            e8_unpack(v, a, b);
            return e8_dec(q, a, b, (float)raw);
        } else {
            float vx, vy;
            Vel<S>::unpack(v, vx, vy);
            return eq_shift(q, vx, vy) + (float)raw;
        }
    }
    static __device__ __forceinline__ float ldh(const Params &p, const s_t *b, int q, size_t c)
    {
        return dec(q, b[(size_t)q * p.N + c], vel(b, p.N)[c]);
    }
    static __device__ __forceinline__ T ld(const Params &p, const s_t *b, int q, size_t c)
    {
        return weight<float>(q) + ldh(p, b, q, c);
    }
};
template <> struct Store<LBM_STORE_F16E> : StoreShifted<LBM_STORE_F16E> {};
template <> struct Store<LBM_STORE_F16E8> : StoreShifted<LBM_STORE_F16E8> {};

__host__ __device__ constexpr bool shifted(int S)
{
    return S == LBM_STORE_F16E || S == LBM_STORE_F16E8;
}

__device__ __forceinline__ int node_x(const Params &p, int cell)
{
    int x = (int)__umulhi((uint32_t)cell, p.magic);
    if (cell - x * p.ny < 0) --x;  // the estimate is never low, at most one high
    return x;
}

__device__ __forceinline__ int bc_row(const Params &p)
{
    int r = (*p.base + p.k) % p.ring;
    return r < 0 ? r + p.ring : r;
}

__device__ __forceinline__ void link_range(const Params &p, int cell, int &lo, int &hi)
{
    lo = hi = 0;
    if (!p.tile_slot) return;
    const int slot = p.tile_slot[cell >> p.tile_shift];
    if (slot < 0) return;
    const int tc = 1 << p.tile_shift;
    const int *off = p.cell_off + (size_t)slot * (tc + 1) + (cell & (tc - 1));
    lo = off[0];
    hi = off[1];
}

template <int S>
__device__ __forceinline__ void pull_checked(const Params &p, int x, int y,
                                             typename Store<S>::T *f)
{
    using St = Store<S>;
    using T = typename St::T;
    const auto *src = static_cast<const typename St::s_t *>(p.src);
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const int sx = x - CX[q], sy = y - CY[q];
        f[q] = (sx >= 0 && sx < p.nx && sy >= 0 && sy < p.ny)
                   ? St::ld(p, src, q, (size_t)sx * p.ny + sy)
                   : T(0);
    }
}

// Deviation value h_qb of one link in the float forms.  The two or three
// sources of a link share the weight w_q (planes q and qb are opposite) and
// the interpolation factors sum to one, so f - w obeys the same affine map:
// the rest state bounces back exactly and float-rounded factors cost a
// relative 1e-7 of the deviation, not of w.
template <int S>
__device__ __forceinline__ float link_h(const Params &p, int cell, const LinkRec &L, float &A)
{
    using St = Store<S>;
    const auto *src = static_cast<const typename St::s_t *>(p.src);
    A = St::ldh(p, src, L.q, cell);
    if (!L.mode) return A;
    const float B = St::ldh(p, src, L.planeB, L.cellB);
    const float C = St::ldh(p, src, L.planeC, L.cellC);
    return ((float)L.c0 * A + (float)L.c1 * B) + (float)L.c2 * C;
}

// Obstacle links of a node on full populations f (nb.py:77-117): f[qb] of
// every link of `cell` (links lo..hi-1).
template <int S>
__device__ __forceinline__ void apply_links(const Params &p, int cell, int lo, int hi,
                                            typename Store<S>::T *f)
{
    using St = Store<S>;
    using T = typename St::T;
    const auto *src = static_cast<const typename St::s_t *>(p.src);
    for (int k = lo; k < hi; ++k) {
        const LinkRec L = p.links[k];
        T v;
        if constexpr (S == LBM_STORE_F64) {
            const T A = St::ld(p, src, L.q, cell);
            v = A;
            if (L.mode) {
                const T B = St::ld(p, src, L.planeB, L.cellB);
                const T C = St::ld(p, src, L.planeC, L.cellC);
                v = (T(L.c0) * A + T(L.c1) * B) + T(L.c2) * C;
            }
        } else {
            float A;
            v = weight<float>(L.qb) + link_h<S>(p, cell, L, A);
        }
        // f[L.qb] = v with a register-resident array
#pragma unroll
        for (int q = 1; q < 9; ++q)
            if (q == L.qb) f[q] = v;
    }
}

// The same on deviations h (float forms, interior nodes).
template <int S>
__device__ __forceinline__ void apply_links_h(const Params &p, int cell, int lo, int hi,
                                              float *h)
{
    for (int k = lo; k < hi; ++k) {
        const LinkRec L = p.links[k];
        float A;
        const float v = link_h<S>(p, cell, L, A);
#pragma unroll
        for (int q = 1; q < 9; ++q)
            if (q == L.qb) h[q] = v;
    }
}

// Wall input `side` of iteration row, element i (component-major, as the
// reference's u_left[2][ny] etc.).  Pool form: a table of wall arrays per
// iteration.  Separable form (batched cases): amplitude(row, side) x profile,
// the reference apps' (ret*u_lbm) * profile_j values.
__device__ __forceinline__ double side_value(const Params &p, int row, int side, int i)
{
    if (p.amp) return p.amp[(size_t)row * p.amp_stride + side] * p.prof[side][i];
    return p.pool[p.inlet_off[row * 5 + side] + i];
}

// Post-boundary populations of a node that is not a domain corner; r, ux, uy
// receive what the wall routine writes to rho/u (perimeter nodes only).
template <int S>
__device__ void gather_edge(const Params &p, int x, int y, int cell, int row,
                            typename Store<S>::T *f, typename Store<S>::T &r,
                            typename Store<S>::T &ux, typename Store<S>::T &uy)
{
    using T = typename Store<S>::T;
    pull_checked<S>(p, x, y, f);
    int lo, hi;
    link_range(p, cell, lo, hi);
    apply_links<S>(p, cell, lo, hi, f);
    const int lx = p.nx - 1, ly = p.ny - 1;
    if (y == 0 && p.bc_bottom) {
        ux = T(side_value(p, row, LBM_SIDE_BOTTOM, x));
        uy = T(side_value(p, row, LBM_SIDE_BOTTOM, p.nx + x));
        zh_bottom(f, ux, uy, r);
    } else if (y == ly && p.bc_top) {
        ux = T(side_value(p, row, LBM_SIDE_TOP, x));
        uy = T(side_value(p, row, LBM_SIDE_TOP, p.nx + x));
        zh_top(f, ux, uy, r);
    } else if (x == 0 && p.bc_left) {
        ux = T(side_value(p, row, LBM_SIDE_LEFT, y));
        uy = T(side_value(p, row, LBM_SIDE_LEFT, p.ny + y));
        zh_left(f, ux, uy, r);
    } else if (x == lx && p.bc_right == LBM_BC_VELOCITY) {
        ux = T(side_value(p, row, LBM_SIDE_RIGHT, y));
        uy = T(side_value(p, row, LBM_SIDE_RIGHT, p.ny + y));
        zh_right_vel(f, ux, uy, r);
    } else if (x == lx && p.bc_right == LBM_BC_PRESSURE) {
        r = T(side_value(p, row, LBM_SIDE_RHO_RIGHT, y));
        uy = T(side_value(p, row, LBM_SIDE_RIGHT, p.ny + y));
        zh_right_pres(f, r, uy, ux);
    }
}

// Post-boundary populations of any node (corners recompute the adjacent
// top/bottom wall node, whose rho/u the reference corner routines copy).
template <int S>
__device__ void gather_bc(const Params &p, int x, int y, int cell, int row,
                          typename Store<S>::T *f, typename Store<S>::T &r,
                          typename Store<S>::T &ux, typename Store<S>::T &uy)
{
    using T = typename Store<S>::T;
    const int lx = p.nx - 1, ly = p.ny - 1;
    const bool xe = (x == 0 || x == lx), ye = (y == 0 || y == ly);
    if (!(xe && ye) || !p.corners) {
        gather_edge<S>(p, x, y, cell, row, f, r, ux, uy);
        return;
    }
    // corner: own streamed populations and links, then the corner routine
    pull_checked<S>(p, x, y, f);
    int lo, hi;
    link_range(p, cell, lo, hi);
    apply_links<S>(p, cell, lo, hi, f);
    const int nxn = (x == 0) ? 1 : lx - 1;
    const int which = (x == 0) ? (y == 0 ? 0 : 1) : (y == 0 ? 3 : 2);
    T fn[9];
    gather_edge<S>(p, nxn, y, nxn * p.ny + y, row, fn, r, ux, uy);
    zh_corner(f, which, r, ux, uy);
}

// Drag ring entry of every link of `cell`: f_q(x) + f_qb(x), the pair the
// momentum exchange sums (nb.py:49-73), in double.  The float forms add the
// exact double weights to the deviations, so the weights cancel over an
// obstacle as they do in FP64.
template <int S>
__device__ __forceinline__ void store_drag_range(const Params &p, int cell, int row, int lo,
                                                 int hi, const typename Store<S>::T *f)
{
    using St = Store<S>;
    const auto *src = static_cast<const typename St::s_t *>(p.src);
    for (int k = lo; k < hi; ++k) {
        const LinkRec L = p.links[k];
        double v;
        if constexpr (S == LBM_STORE_F64) {
            double fb = 0.0;
#pragma unroll
            for (int q = 1; q < 9; ++q)
                if (q == L.qb) fb = f[q];
            v = St::ld(p, src, L.q, cell) + fb;
        } else {
            // f[qb] = fl(w + h) with |h| < w/2, so f[qb] - w is exact (Sterbenz)
            float hb = 0.0f;
#pragma unroll
            for (int q = 1; q < 9; ++q)
                if (q == L.qb) hb = f[q] - weight<float>(q);
            const double hA = (double)St::ldh(p, src, L.q, cell);
            v = 2.0 * weight<double>(L.q) + (hA + (double)hb);
        }
        p.drag_ring[(size_t)row * p.n_links + L.dslot] = v;
    }
}

// The same from deviations h (float forms, interior nodes).
template <int S>
__device__ __forceinline__ void store_drag_range_h(const Params &p, int cell, int row, int lo,
                                                   int hi, const float *h)
{
    using St = Store<S>;
    const auto *src = static_cast<const typename St::s_t *>(p.src);
    for (int k = lo; k < hi; ++k) {
        const LinkRec L = p.links[k];
        float hb = 0.0f;
#pragma unroll
        for (int q = 1; q < 9; ++q)
            if (q == L.qb) hb = h[q];
        const double hA = (double)St::ldh(p, src, L.q, cell);
        p.drag_ring[(size_t)row * p.n_links + L.dslot] =
            2.0 * weight<double>(L.q) + (hA + (double)hb);
    }
}

template <int S>
__device__ __forceinline__ void store_drag(const Params &p, int cell, int row,
                                           const typename Store<S>::T *f)
{
    int lo, hi;
    link_range(p, cell, lo, hi);
    store_drag_range<S>(p, cell, row, lo, hi, f);
}

// Moments, equilibrium and TRT collision (lattice.py:178-189, nb.py:7-17,
// nb.py:24-35): o = post-collision populations of the post-boundary f.
__device__ __forceinline__ void collide_f64(const Params &p, const double *f, double *o, double &r,
                                            double &ux, double &uy)
{
    r = f[0];
#pragma unroll
    for (int q = 1; q < 9; ++q) r = r + f[q];
    const double sx = ((((f[1] - f[2]) + f[5]) - f[6]) - f[7]) + f[8];
    const double sy = ((((f[3] - f[4]) + f[5]) - f[6]) + f[7]) - f[8];
    ux = sx / r;
    uy = sy / r;
    // g_eq of nb.py:13-17, (1 + t + t^2 / 2 - v) (rho w) with t = 3 c.u.  t of
    // an opposite direction is -t, exactly: the pair shares t and its square.
    const double v = 1.5 * (ux * ux + uy * uy);
    const double zx = ux * 0.0, zy = uy * 0.0;   // c = 0 terms (NaN for a non-finite u)
    const double t0 = 3.0 * (zx + zy);
    o[0] = p.b0 * f[0] + p.om_p * ((1.0 + t0 + 0.5 * (t0 * t0) - v) * (r * weight<double>(0)));
#pragma unroll
    for (int q = 1; q < 9; q += 2) {             // pairs (1,2) (3,4) (5,6) (7,8)
        const double t = 3.0 * (q == 1   ? ux + zy
                                : q == 3 ? zx + uy
                                : q == 5 ? ux + uy
                                         : uy - ux);
        const double s = 0.5 * (t * t), rw = r * weight<double>(q);
        const double e = (1.0 + t + s - v) * rw, eb = (1.0 - t + s - v) * rw;
        o[q] = p.a1 * f[q] - p.a2 * f[q + 1] + p.a3 * e + p.a4 * eb;
        o[q + 1] = p.a1 * f[q + 1] - p.a2 * f[q] + p.a3 * eb + p.a4 * e;
    }
}

template <int S>
__device__ __forceinline__ void collide_store(const Params &p, int cell,
                                              typename Store<S>::T *f, bool macro)
{
    static_assert(S == LBM_STORE_F64, "the float forms collide deviations (collide_store_h)");
    double *dst = static_cast<double *>(p.dst);
    double o[9], r, ux, uy;
    collide_f64(p, f, o, r, ux, uy);
    if (macro) {
        p.rho_out[cell] = r;
        p.u_out[cell] = ux;
        p.u_out[(size_t)p.N + cell] = uy;
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) dst[(size_t)q * p.N + cell] = o[q];
}

// Float forms: moments, equilibrium and TRT collision on the deviations
// h_q = f_q - w_q, with the collision written per opposite pair (q, qb):
//   h+- = (h_q +- h_qb)/2,  E+ = w (drho + rho (4.5 cu^2 - 1.5 u^2)),
//   E- = 3 w rho cu,  h_q' = h_q - om_p (h+ - E+) - om_m (h- - E-),
//   h_qb' = h_qb - om_p (h+ - E+) + om_m (h- - E-),
// which is nb.py:24-35 with g_eq of nb.py:7-17, rearranged (E = g_eq - w).
struct Coll {
    float op, hp, hm;  // om_p, om_p/2, om_m/2
};

__device__ __forceinline__ Coll coll_consts(const Params &p)
{
    return Coll{p.omf_p, 0.5f * p.omf_p, 0.5f * p.omf_m};
}

// In place: h (deviations of one node) -> post-collision deviations.
// Every multiply-add is an explicit fmaf and nothing else is contracted (the
// library builds with -ffp-contract=off), so each kernel that inlines this
// -- one node per lane, four nodes per lane, batched -- rounds identically.
__device__ __forceinline__ void collide_h(const Coll &k, float *h, float &rho, float &ux,
                                          float &uy)
{
    const float drho = ((h[0] + h[1]) + (h[2] + h[3])) + ((h[4] + h[5]) + (h[6] + h[7])) + h[8];
    const float d78 = h[7] - h[8];
    const float jx = (h[1] - h[2]) + (h[5] - h[6]) - d78;
    const float jy = (h[3] - h[4]) + (h[5] - h[6]) + d78;
    rho = 1.0f + drho;
    const float inv = __builtin_amdgcn_rcpf(rho);
    ux = jx * inv;
    uy = jy * inv;
    const float usq = 1.5f * __builtin_fmaf(uy, uy, ux * ux);
    const float base = __builtin_fmaf(-rho, usq, drho);   // E+/w without the 4.5 cu^2 term
    const float e0 = weight<float>(0) * base;
    h[0] = __builtin_fmaf(-k.op, h[0] - e0, h[0]);
    const float wr3[2] = {3.0f * weight<float>(1) * rho, 3.0f * weight<float>(5) * rho};
    const float w45[2] = {4.5f * weight<float>(1) * rho, 4.5f * weight<float>(5) * rho};
    const float wb[2] = {weight<float>(1) * base, weight<float>(5) * base};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int q = 2 * j + 1, qb = q + 1;   // pairs (1,2) (3,4) (5,6) (7,8)
        const int d = j < 2 ? 0 : 1;
        const float cu = j == 0 ? ux : (j == 1 ? uy : (j == 2 ? ux + uy : uy - ux));
        const float ep = __builtin_fmaf(w45[d] * cu, cu, wb[d]);
        const float em = wr3[d] * cu;
        const float dp = k.hp * __builtin_fmaf(-2.0f, ep, h[q] + h[qb]);
        const float dm = k.hm * __builtin_fmaf(-2.0f, em, h[q] - h[qb]);
        const float a = (h[q] - dp) - dm;
        const float bb = (h[qb] - dp) + dm;
        h[q] = a;
        h[qb] = bb;
    }
}

template <int S>
__device__ __forceinline__ void collide_store_h(const Params &p, int cell, const float *hin,
                                                bool macro)
{
    using St = Store<S>;
    auto *dst = static_cast<typename St::s_t *>(p.dst);
    float h[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) h[q] = hin[q];
    float rho, ux, uy;
    collide_h(coll_consts(p), h, rho, ux, uy);
    if (macro) {
        p.rho_out[cell] = (double)rho;
        p.u_out[cell] = (double)ux;
        p.u_out[(size_t)p.N + cell] = (double)uy;
    }
    if constexpr (shifted(S)) {
        // the node's velocity word, then g_q = h_q - E_q(v) of the stored v
        using w_t = typename Vel<S>::w_t;
        const uint32_t off = (uint32_t)cell * (uint32_t)sizeof(typename St::s_t);
        if constexpr (S == LBM_STORE_F16E8) {
            float a, b;
            st_off(sbase(dst + vel_offset(p.N)), off, e8_pack(ux, uy, a, b));
#pragma unroll
            for (int q = 0; q < 9; ++q)
                st_off(sbase(dst + (size_t)q * p.N), off, to_half(h[q] - e8_shift(q, a, b)));
        } else {
            const w_t v = Vel<S>::pack(ux, uy);
            reinterpret_cast<w_t *>(dst + vel_offset(p.N))[cell] = v;
            float vx, vy;
            Vel<S>::unpack(v, vx, vy);
#pragma unroll
            for (int q = 0; q < 9; ++q)
                st_off(sbase(dst + (size_t)q * p.N), off, to_half(h[q] - eq_shift(q, vx, vy)));
        }
    } else if constexpr (is16(S)) {
        const uint32_t off = (uint32_t)cell * (uint32_t)sizeof(typename St::s_t);
#pragma unroll
        for (int q = 0; q < 9; ++q) st_off(sbase(dst + (size_t)q * p.N), off, St::enc(p, q, h[q]));
    } else {
#pragma unroll
        for (int q = 0; q < 9; ++q) St::sth(p, dst, q, (size_t)q * p.N + cell, h[q]);
    }
}

// Work-group index -> tile index, so that each XCD (work-groups are dealt
// round-robin over the 8 XCDs) sweeps one contiguous slab of the lattice and
// the rows its tiles share stay in that XCD's L2 (the multi-iteration tiles;
// the one-iteration step sweeps its tiles in dispatch order, sweep_tile).
// With rev set the slab is swept last tile first.
__device__ __forceinline__ int xcd_tile(int b, int nb, int rev = 0)
{
    const int q = nb >> 3, rr = nb & 7;
    const int xcd = b & 7, i = b >> 3;
    const int len = q + (xcd < rr ? 1 : 0);   // work-groups of this XCD
    return xcd * q + min(xcd, rr) + (rev ? len - 1 - i : i);
}

template <int S>
__device__ __forceinline__ void collide_any(const Params &p, int cell,
                                            typename Store<S>::T *f, bool macro)
{
    if constexpr (S == LBM_STORE_F64) {
        collide_store<S>(p, cell, f, macro);
    } else {
        float h[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) h[q] = f[q] - weight<float>(q);
        collide_store_h<S>(p, cell, h, macro);
    }
}

// One word of every 64-byte line of a parameter block, loaded in one batch:
// the fields a kernel reads are otherwise fetched in several dependent rounds
// of scalar loads, each of which can miss the scalar cache.  The batched step
// reads each work item's block from device memory and gains from it (256
// cavities, FP32: 62.8 -> 65.3 GLUPS); the one-lattice step reads its block
// from the kernel arguments and does not (f16e8 on the 8192x2048 obstacle
// array: 143 -> 150 us with it).
__device__ __forceinline__ void touch_params(const Params &p)
{
    const uint32_t *w = reinterpret_cast<const uint32_t *>(&p);
    constexpr int lines = (int)((sizeof(Params) + 63) / 64);
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < lines; ++i) acc ^= w[i * 16];
    asm volatile("" ::"s"(acc));
}

}  // namespace lbm
