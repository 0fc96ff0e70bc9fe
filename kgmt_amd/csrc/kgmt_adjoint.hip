// kgmt_adjoint.hip — differentiable RK4 rollout of the quadcopter ODE on gfx950.
//
// Refinement of found control sequences (an extension beside the planner).
// A trajectory integrates x_{t+1} = RK4(x_t, u_t) forward and runs the
// discrete adjoint of those steps backward. The cost is
//   J = w_e sum |u_t - u_ref|^2 + w_o sum_{t>=1} sum_b tau softplus((m - sd(p_t, b)) / tau)
//     + w_g |p_T - goal|^2.
// k_rollout<false> writes J and dJ/du; k_rollout<true> runs Adam for
// `iterations` steps in place and records J before every step and after the
// last. The dynamics are those of statePropagator.cu:325-370 (ode).
//
// What bounds it: the time steps form a chain, and a wave issues at most one
// vector instruction every 4 cycles, so the time of a pass is the number of
// instructions on the chain. Only what must follow the chain stays on it:
//   1. forward chain: attitude and body velocities. The position feeds back
//      into nothing, so it is left out. Lane c of a quad carries component c
//      of the angles, the body velocity and the body rates; one sin/cos, one
//      cross product and one square root serve all three components, and a
//      step takes a quarter of the instructions that one lane would need. The
//      four stages' states are kept for the passes below.
//   2. positions, penalties and J, lane = (step, stage): the stages' world
//      velocities, their sum over a step by quad permutations, a scan over
//      groups of four steps and a sum over the groups, then the boxes spread
//      over a step's four lanes.
//   3. backward, lane = (step, stage): the stage's vector-Jacobian product as
//      eight rows of coefficients in LDS (the adjoints of the positions and of
//      psi do not depend on the others: suffix sums over the steps, folded
//      into the rows' constants), then the backward chain: lane j of a row of
//      16 lanes holds adjoint j, and a stage is eight multiply-adds with
//      broadcast operands.
// The kernel that ran the whole step in every lane of a trajectory took
// 47.2 ms for 4096 trajectories (20..80 steps, 50 Adam steps, 50 boxes),
// 1.28 ms for one cost and gradient of them and 1.51 ms for 333 trajectories
// among 301 boxes; this one takes 7.78, 0.23 and 0.13 ms, and its error
// against 64 bits is smaller (gradient of the 333: 2.4e-6 to 2.7e-7).
#include <algorithm>

#include "kgmt_launch.hpp"

// Within an expression: which products are fused follows from the source
// alone, so the kernel has the same bits for every number of lanes.
#pragma clang fp contract(on)

namespace kgmt
{

namespace
{

// sin and cos as sincos_k (the same reduction and polynomials) with fused
// multiply-adds
__device__ __forceinline__ void sincos_fused(float x, float& s, float& c)
{
    const float fk = __builtin_rintf(x * 0x1.45f306p-1f);
    float r        = __builtin_fmaf(-fk, 0x1.92p+0f, x);
    r              = __builtin_fmaf(-fk, 0x1.fb4p-12f, r);
    r              = __builtin_fmaf(-fk, 0x1.4442d2p-24f, r);
    const int m    = (int)fk;
    const float z  = r * r;
    float ps       = __builtin_fmaf(0x1.71de3ap-19f, z, -0x1.a01a02p-13f);
    ps             = __builtin_fmaf(ps, z, 0x1.111112p-7f);
    ps             = __builtin_fmaf(ps, z, -0x1.555556p-3f);
    const float sr = __builtin_fmaf(r * z, ps, r);
    float pc       = __builtin_fmaf(0x1.1eed8ep-29f, z, -0x1.27e4fcp-22f);
    pc             = __builtin_fmaf(pc, z, 0x1.a01a02p-16f);
    pc             = __builtin_fmaf(pc, z, -0x1.6c16c2p-10f);
    pc             = __builtin_fmaf(pc, z, 0x1.555556p-5f);
    const float cr = __builtin_fmaf(z * z, pc, __builtin_fmaf(-0.5f, z, 1.0f));
    const float a  = (m & 1) ? cr : sr;
    const float b  = (m & 1) ? sr : cr;
    s              = (m & 2) ? -a : a;
    c              = ((m + 1) & 2) ? -b : b;
}

// (s, c) turned by the small angle d (|d| < 0.1: the series' first term left
// out is below 3e-10)
__device__ __forceinline__ void turn(float s0, float c0, float d, float& s, float& c)
{
    const float z  = d * d;
    const float sd = __builtin_fmaf(d * z, __builtin_fmaf(z, 1.0f / 120.0f, -1.0f / 6.0f), d);
    const float cm = z * __builtin_fmaf(z, __builtin_fmaf(z, -1.0f / 720.0f, 1.0f / 24.0f), -0.5f);  // cos d - 1
    s              = __builtin_fmaf(c0, sd, __builtin_fmaf(s0, cm, s0));
    c              = __builtin_fmaf(-s0, sd, __builtin_fmaf(c0, cm, c0));
}

// 1 / x within one ulp
__device__ __forceinline__ float recip(float x)
{
    return __builtin_amdgcn_rcpf(x);
}

// v of the lane that the DPP control selects (every control used here stays
// inside the row)
template <int CTRL>
__device__ __forceinline__ float dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
constexpr int kQuad0 = 0x00, kQuad1 = 0x55, kQuad2 = 0xAA, kQuad3 = 0xFF;  // quad_perm: one lane to its quad
constexpr int kNext  = 0xC9;   // quad_perm [1,2,0,3]: component c + 1 of three
constexpr int kPrev  = 0xD2;   // quad_perm [2,0,1,3]: component c + 2

// y += sum over k < 8 of x of lane k of the row times ck: eight multiply-adds
// that read their broadcast operand by DPP (the compiler keeps a move before
// each). A DPP read needs two wait states after the write of x: the s_nop.
__device__ __forceinline__ void row_madd(float& y, float x, float c0, float c1, float c2, float c3, float c4, float c5,
                                         float c6, float c7)
{
#define KGMT_MADD(K, R) "v_fmac_f32_dpp %0, %1, " R " row_newbcast:" K " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" KGMT_MADD("0", "%2") KGMT_MADD("1", "%3") KGMT_MADD("2", "%4") KGMT_MADD("3", "%5")
          KGMT_MADD("4", "%6") KGMT_MADD("5", "%7") KGMT_MADD("6", "%8") KGMT_MADD("7", "%9")
        : "+&v"(y)  // written before the last operands are read
        : "v"(x), "v"(c0), "v"(c1), "v"(c2), "v"(c3), "v"(c4), "v"(c5), "v"(c6), "v"(c7));
#undef KGMT_MADD
}

// (hi, lo) += v: hi the rounded sum, lo what its roundings left (NaN once hi
// is infinite: known())
__device__ __forceinline__ void add_exact(float& hi, float& lo, float v)
{
    const float s = hi + v, b = s - hi;
    lo += (hi - (s - b)) + (v - b);
    hi = s;
}

__device__ __forceinline__ float known(float lo)
{
    return lo == lo ? lo : 0.0f;
}

__device__ __forceinline__ float quad_sum(float v)
{
    v += dpp<0xB1>(v);
    return v + dpp<0x4E>(v);
}

// four values per lane -> lane c of the quad holds the quad's sum of v[c]
__device__ __forceinline__ float quad_scatter(const float (&v)[4], int lane)
{
    const bool b1 = lane & 2, b0 = lane & 1;
    const float x = (b1 ? v[2] : v[0]) + dpp<0x4E>(b1 ? v[0] : v[2]);
    const float y = (b1 ? v[3] : v[1]) + dpp<0x4E>(b1 ? v[1] : v[3]);
    return (b0 ? y : x) + dpp<0xB1>(b0 ? x : y);
}

// tau * softplus(x / tau), x = margin - sd, of one box at p, and its gradient:
// max(x, 0) + tau log1p(e) and (1 or e) / (1 + e) with e = exp(-|x| / tau);
// log1p(e) = 2 atanh(t), t = e / (2 + e), the polynomial by Chebyshev
// interpolation over t^2 <= 1/9. The root, the reciprocal and the exponential
// of the units are within an ulp; each is followed by the step that takes its
// error out (the residuals of the root and of the quotients, the rest of the
// exponent's product): one box's penalty is 0.7 to 1.05 times as far from 64
// bits as by the library's sqrt, division, expf and log1pf (its gradient 0.75
// to 1.1 times), 1.0 to 2.2 times without. That costs 4 %: refine of 4096
// trajectories among 50 boxes 7.48 to 7.77 ms. acc: half the logarithms, and
// the gradient; flat: the max(x, 0).
__device__ __forceinline__ void box_penalty(float4 lo, float4 hi, float px, float py, float pz, float margin,
                                            float tau, const RolloutK& K, bool plain, uint64_t anyPlain,
                                            float (&acc)[4], float& flat)
{
    const float lx = lo.x - px, hx = px - hi.x, ly = lo.y - py, hy = py - hi.y, lz = lo.z - pz, hz = pz - hi.z;
    const bool nx = lx > hx, ny = ly > hy, nz = lz > hz;  // nearer the low face
    const float qx = nx ? lx : hx, qy = ny ? ly : hy, qz = nz ? lz : hz;
    const float ox = fmaxf(qx, 0.0f), oy = fmaxf(qy, 0.0f), oz = fmaxf(qz, 0.0f);
    const float d2 = ox * ox + oy * oy + oz * oz;
    const float id = __builtin_amdgcn_rsqf(d2), s0 = d2 * id;
    float sd       = __builtin_fmaf(__builtin_fmaf(-s0, s0, d2), 0.5f * id, s0);
    float x        = margin - sd;
    // -|x| / tau in base 2: rounded, and what the rounding leaves
    float y  = -fabsf(x) * K.eHi;
    float yl = __builtin_fmaf(-fabsf(x), K.eLo, __builtin_fmaf(-fabsf(x), K.eHi, -y));
    // outside: (ox, oy, oz) / distance; inside: the axis of the nearest face,
    // the first of the largest. The unit's reciprocal root holds for normal d2
    // alone: a face or a corner within 1e-19 and a box farther than 1.8e19
    // take a scaled root, as inside does, and the plain quotient by tau (rare:
    // one vote of the active lanes skips it; the other lanes keep what they
    // have; plain: a position or a scene that is not finite, or tau or margin
    // out of the range of the short form)
    float vx = ox * id, vy = oy * id, vz = oz * id;
    const bool edge = __builtin_amdgcn_classf(d2, 0x2ff);  // not a positive normal
    if((__builtin_amdgcn_ballot_w64(edge) | anyPlain) != 0u)
        {
            const bool odd  = plain | edge;
            const bool tiny = !(d2 >= 0x1p-126f), huge = !(d2 <= 0x1.fffffep127f);
            const float k  = tiny ? 0x1p100f : huge ? 0x1p-100f : 1.0f;
            const float rk = tiny ? 0x1p-100f : huge ? 0x1p100f : 1.0f;
            const float kx = ox * k, ky = oy * k, kz = oz * k;
            const float root = __builtin_sqrtf(kx * kx + ky * ky + kz * kz), len = root * rk;
            const float ux = kx / root, uy = ky / root, uz = kz / root;
            const bool out = root > 0.0f;
            const bool xy = qx >= qy, ax = xy & (qx >= qz), ay = !xy & (qy >= qz);
            sd = odd ? (out ? len : 0.0f) + fminf(ax ? qx : ay ? qy : qz, 0.0f) : sd;
            vx = odd ? (out ? ux : ax ? 1.0f : 0.0f) : vx;
            vy = odd ? (out ? uy : ay ? 1.0f : 0.0f) : vy;
            vz = odd ? (out ? uz : (ax | ay) ? 0.0f : 1.0f) : vz;
            x  = margin - sd;
            const float z = fabsf(x / tau), c = z > 110.0f ? 110.0f : z;  // (e^-104 is 0; NaN stays)
            const float w = c * -0x1.715476p+0f;
            yl = odd ? __builtin_fmaf(c, -0x1.4ae0cp-26f, __builtin_fmaf(c, -0x1.715476p+0f, -w)) : yl;
            y  = odd ? w : y;
        }
    const float e0 = __builtin_amdgcn_exp2f(y), e = __builtin_fmaf(e0, 0.693147181f * yl, e0);
    // one reciprocal for 1 / (2 + e) and 1 / (1 + e)
    const float e1 = 1.0f + e, e2 = 2.0f + e, el = e - (e2 - 2.0f);
    const float re = recip(e1 * e2), r1 = e2 * re, r2 = e1 * re;
    const float t0 = e * r2, tr = __builtin_fmaf(-t0, el, __builtin_fmaf(-t0, e2, e)) * r2, t = t0 + tr, u = t * t;
    float at       = __builtin_fmaf(u, 0x1.dba25ep-4f, 0x1.bc8cf8p-4f);
    at             = __builtin_fmaf(u, at, 0x1.24c926p-3f);
    at             = __builtin_fmaf(u, at, 0x1.9998d4p-3f);
    at             = __builtin_fmaf(u, at, 0x1.555556p-2f);
    acc[0]         = __builtin_fmaf(tau, t0 + __builtin_fmaf(t * u, at, tr), acc[0]);  // (half of it)
    const bool up  = x >= 0.0f;
    flat += up ? x : 0.0f;
    const float n  = up ? 1.0f : e;
    const float g0 = n * r1, g = __builtin_fmaf(__builtin_fmaf(-g0, e1, n), r1, g0);
    acc[1]         = __builtin_fmaf(nx ? g : -g, vx, acc[1]);
    acc[2]         = __builtin_fmaf(ny ? g : -g, vy, acc[2]);
    acc[3]         = __builtin_fmaf(nz ? g : -g, vz, acc[3]);
}

constexpr int kRowWords   = 12;   // a row of coefficients: constant, then those of a3 a4 a6 a7 a8 a9 a10 a11
constexpr int kBlockWords = 100;  // eight rows of one (step, stage), padded: 16 lanes' blocks start in distinct banks
constexpr int kStageWords = 48;   // kept per step: angles, velocity, rates, each [4 stages][4]

// box slots of the LDS for n boxes: the next four of a lane's last box fit
__host__ __device__ constexpr uint32_t box_slots(uint32_t n)
{
    return n + 8;
}

struct RolloutLds
{
    float coef[64 * kBlockWords];
    float ubar[64];
};

}  // namespace

// LPT lanes per trajectory (64 / LPT trajectories per wave, one wave per
// workgroup); LPT / 4 steps per round of passes 2 and 3. work: per trajectory
// of this launch maxT * (kStageWords + 8 [+ 8]) floats: stage states, per step
// the penalty, its gradient and the controls, and, when refining, the Adam
// moments. (The controls are copied first: the caller's layout puts a
// trajectory's steps 16 n bytes apart, a page each, and the chain would wait
// for each of them.)
template <bool REFINE, int LPT>
__global__ __launch_bounds__(64) void k_rollout(RolloutK K, kgmt_adjoint_params ap, uint32_t i0, uint32_t n,
                                                uint32_t maxT, const int32_t* __restrict__ steps,
                                                const float* __restrict__ x0g, const float* __restrict__ goalg,
                                                float* u, float* __restrict__ grad, float* work,
                                                const float* __restrict__ rows, uint32_t nObs,
                                                float* __restrict__ cost)
{
    constexpr int CH = LPT / 4;  // steps per round
    extern __shared__ float4 sBox[];  // low corners, then high corners
    __shared__ RolloutLds L;
    const int lane = (int)threadIdx.x;
    const uint32_t nBox = box_slots(nObs);  // the read ahead ends inside the slots (unused ones hold anything)
    bool odd            = K.plain != 0u;
    for(uint32_t k = lane; k < nObs; k += 64)
        {
            const float* r = rows + 6 * (size_t)k;
            const float4 lo = make_float4(r[0], r[1], r[2], 0.0f), hi = make_float4(r[3], r[4], r[5], 0.0f);
            sBox[k]        = lo;
            sBox[nBox + k] = hi;
            // (0 x: NaN unless x is finite)
            const float f = 0.0f * lo.x + 0.0f * lo.y + 0.0f * lo.z + 0.0f * hi.x + 0.0f * hi.y + 0.0f * hi.z;
            odd |= f != 0.0f;
        }
    const bool scenePlain = __any(odd);
    __syncthreads();
    const uint32_t slot = (blockIdx.x * 64 + lane) / LPT;
    const uint32_t i    = i0 + slot < n ? i0 + slot : n - 1;  // lanes past the end read the last trajectory
    const bool act      = i0 + slot < n;                      // and write nothing
    const int l         = lane % LPT;
    const int tt = l >> 2, s = l & 3;  // passes 2 and 3: step of the round, stage (or control)
    const int j  = l & 7;              // backward chain: row
    const int gb = lane - l;           // first lane of the trajectory
    const size_t N = n;
    int T          = act ? steps[i] : 0;
    T              = T < 0 ? 0 : (T > (int)maxT ? (int)maxT : T);
    int Tm         = T;  // longest of the wave
#pragma unroll
    for(int o = LPT; o < 64; o <<= 1)
        {
            const int x = __shfl_xor(Tm, o, 64);
            Tm          = x > Tm ? x : Tm;
        }
    Tm             = __builtin_amdgcn_readfirstlane(Tm);
    float* W       = work + (size_t)slot * maxT * (kStageWords + 8 + (REFINE ? 8 : 0));
    float* Wg      = W + (size_t)maxT * kStageWords;  // penalty (0) and its gradient (1..3) at x_{t+1}, u_t (4..7)
    float* Wm      = Wg + (size_t)maxT * 8;           // moments [t][4] x 2
    const float gx = goalg[i], gy = goalg[N + i], gz = goalg[2 * N + i];
    const float p0x = x0g[i], p0y = x0g[N + i], p0z = x0g[2 * N + i];
    const int c3     = s < 3 ? s : 2;  // forward chain: component of this lane (lane 3 repeats lane 2)
    const float A0 = x0g[(3 + c3) * N + i], U0 = x0g[(6 + c3) * N + i], P0 = x0g[(9 + c3) * N + i];
    const float qa = s == 0 ? K.ax : s == 1 ? K.ay : K.az, qb = s == 0 ? K.bx : s == 1 ? K.by : K.bz;
    const float uref   = s == 0 ? ap.u_ref[0] : s == 1 ? ap.u_ref[1] : s == 2 ? ap.u_ref[2] : ap.u_ref[3];
    const float uscale = s == 0 ? K.minv : s == 1 ? K.bx : s == 2 ? K.by : K.bz;
    const float umin   = s == 0 ? K.cmin[0] : s == 1 ? K.cmin[1] : s == 2 ? K.cmin[2] : K.cmin[3];
    const float umax   = s == 0 ? K.cmax[0] : s == 1 ? K.cmax[1] : s == 2 ? K.cmax[2] : K.cmax[3];
    const float hS     = s == 0 || s == 3 ? K.h6 : K.h3;  // weight of stage s in the step
    const float* uF    = Wg + 4 + ((s + 1) & 3);  // forward: lane c takes control c + 1, lane 3 control 0
    const uint32_t iters = REFINE ? ap.iterations : 0;
    for(int t0 = 0; t0 < Tm; t0 += 4 * CH)
        {
            float x[4];
#pragma unroll
            for(int k = 0; k < 4; ++k)
                {
                    const int t = t0 + k * CH + tt;
                    x[k]        = t < T ? u[((size_t)t * 4 + s) * N + i] : 0.0f;  // (rows past the length are not read)
                }
#pragma unroll
            for(int k = 0; k < 4; ++k)
                {
                    const int t = t0 + k * CH + tt;
                    if(t < Tm) Wg[(size_t)t * 8 + 4 + s] = x[k];
                }
        }
    __threadfence_block();
    float b1t = 1.0f, b2t = 1.0f;
    for(uint32_t it = 0; it <= iters; ++it)
        {
            // 1. forward chain
            {
                float A = A0, U = U0, P = P0;
                const float gd = -K.minv * K.nu, wd = -qb * K.mu;
                float un = Tm > 0 ? uF[0] : 0.0f;
                for(int t = 0; t < Tm; ++t)
                    {
                        const bool on  = LPT == 64 || t < T;  // else the state stays as it is
                        const float uc = un;
                        if(t + 1 < Tm) un = uF[(size_t)(t + 1) * 8];
                        const float u0  = dpp<kQuad3>(uc);
                        const float thr = s == 2 ? K.minv * u0 : 0.0f;
                        const float tor = qb * uc;
                        auto deriv = [&](float sn, float cs, float v, float w, float& da, float& dv, float& dw) {
                            const float sph = dpp<kQuad0>(sn), cph = dpp<kQuad0>(cs);
                            const float sth = dpp<kQuad1>(sn), cth = dpp<kQuad1>(cs);
                            const float v1 = dpp<kNext>(v), v2 = dpp<kPrev>(v);
                            const float w1 = dpp<kNext>(w), w2 = dpp<kPrev>(w);
                            const float q = dpp<kQuad1>(w), r = dpp<kQuad2>(w);
                            const float Ei = (q * sph + r * cph) * recip(cth);
                            const float F  = q * cph - r * sph;
                            da             = s == 0 ? w + Ei * sth : s == 1 ? F : Ei;
                            const float gv = s == 0 ? -sth : cth * (s == 1 ? sph : cph);
                            const float nv = __builtin_amdgcn_sqrtf(v * v + v1 * v1 + v2 * v2);
                            dv = (w2 * v1 - w1 * v2) + K.g * gv + thr + gd * nv * v;
                            const float nw = __builtin_amdgcn_sqrtf(w * w + w1 * w1 + w2 * w2);
                            dw = qa * w1 * w2 + wd * nw * w + tor;
                        };
                        float a1, v1, w1, a2, v2, w2, a3, v3, w3, a4, v4, w4;
                        // the stages' angles are the step's, turned by what
                        // they advance (a fast spin or a long step: past
                        // 0.1 rad sin / cos of the stage's angle; each lane
                        // by its own angle, whatever the others of the wave
                        // hold, so that a trajectory's bits are its own)
                        float sn0, cs0, sn, cs;
                        sincos_fused(A, sn0, cs0);
                        auto angle = [&](float d) {
                            const bool wide = !(fabsf(d) < 0.1f);
                            turn(sn0, cs0, d, sn, cs);
                            if(__any(wide))
                                {
                                    float s1, c1;
                                    sincos_fused(A + d, s1, c1);
                                    sn = wide ? s1 : sn, cs = wide ? c1 : cs;
                                }
                        };
                        // quad k of the row keeps stage k's state
                        const int quad = (l >> 2) & 3;
                        float kA = A, kU = U, kP = P, d, sv, sw;
                        deriv(sn0, cs0, U, P, a1, v1, w1);
                        d = K.hh * a1, sv = U + K.hh * v1, sw = P + K.hh * w1;
                        angle(d);
                        kA = quad == 1 ? A + d : kA, kU = quad == 1 ? sv : kU, kP = quad == 1 ? sw : kP;
                        deriv(sn, cs, sv, sw, a2, v2, w2);
                        d = K.hh * a2, sv = U + K.hh * v2, sw = P + K.hh * w2;
                        angle(d);
                        kA = quad == 2 ? A + d : kA, kU = quad == 2 ? sv : kU, kP = quad == 2 ? sw : kP;
                        deriv(sn, cs, sv, sw, a3, v3, w3);
                        d = K.h * a3, sv = U + K.h * v3, sw = P + K.h * w3;
                        angle(d);
                        kA = quad == 3 ? A + d : kA, kU = quad == 3 ? sv : kU, kP = quad == 3 ? sw : kP;
                        deriv(sn, cs, sv, sw, a4, v4, w4);
                        if(l < 16)
                            {
                                float* o = W + (size_t)t * kStageWords + l;
                                o[0] = kA, o[16] = kU, o[32] = kP;
                            }
                        const float An = A + K.h6 * (a1 + 2.0f * a2 + 2.0f * a3 + a4);
                        const float Un = U + K.h6 * (v1 + 2.0f * v2 + 2.0f * v3 + v4);
                        const float Pn = P + K.h6 * (w1 + 2.0f * w2 + 2.0f * w3 + w4);
                        A = on ? An : A, U = on ? Un : U, P = on ? Pn : P;
                    }
            }
            __threadfence_block();  // the stage states, read by other lanes below
            // 2. positions, penalties, J
            float px = p0x, py = p0y, pz = p0z;  // position at the end of the rounds before
            // Sums over the steps run in fours (16 lanes) one after the other,
            // and J in four parts, step t in part t / 4 % 4, so that a
            // trajectory's bits do not follow from its lanes, which follow
            // from the number of trajectories. The positions carry what
            // the sums' roundings leave (a chain of plain sums is further from
            // 64 bits than a tree: gradient of 333 trajectories among 301
            // boxes 1.3e-6, 7.1e-7 as a tree over 16 steps).
            float rx = 0.0f, ry = 0.0f, rz = 0.0f;
            float Jp[64 / LPT];
#pragma unroll
            for(int k = 0; k < 64 / LPT; ++k) Jp[k] = 0.0f;
            // (each round's reads go out a round ahead)
            const int tl = T > 0 ? T - 1 : 0;
            float4 an, vn;
            float dn = 0.0f;
            auto fetch2 = [&](int t) {
                const int tc     = t < tl ? t : tl;
                const float4* w4 = reinterpret_cast<const float4*>(W + (size_t)tc * kStageWords);
                an = w4[s], vn = w4[4 + s];
                dn = Wg[(size_t)tc * 8 + 4 + s];
            };
            if(Tm > 0) fetch2(tt);
            for(int t0 = 0; t0 < Tm; t0 += CH)
                {
                    const int t    = t0 + tt;
                    const bool on  = t < T;
                    const float4 a = an, v = vn;
                    const float d  = dn - uref;
                    fetch2(t + CH);
                    float sf, cf, st, ct, sp, cp;
                    sincos_fused(a.x, sf, cf);
                    sincos_fused(a.y, st, ct);
                    sincos_fused(a.z, sp, cp);
                    // the velocity turned about x by phi, about y by theta, about z by psi
                    const float m  = sf * v.y + cf * v.z, be = cf * v.y - sf * v.z;
                    const float al = ct * v.x + st * m;
                    float dx = quad_sum(hS * (cp * al - sp * be));
                    float dy = quad_sum(hS * (sp * al + cp * be));
                    float dz = quad_sum(hS * (ct * m - st * v.x));
                    dx = on ? dx : 0.0f, dy = on ? dy : 0.0f, dz = on ? dz : 0.0f;
#pragma unroll
                    for(int o = 4; o < 16; o <<= 1)
                        {
                            const float ex = __shfl_up(dx, o, 16), ey = __shfl_up(dy, o, 16);
                            const float ez = __shfl_up(dz, o, 16);
                            if((l & 15) >= o) dx += ex, dy += ey, dz += ez;
                        }
#pragma unroll
                    for(int g = 16; g < LPT; g += 16)
                        {
                            const float ex = __shfl(dx, g - 1, LPT), ey = __shfl(dy, g - 1, LPT);
                            const float ez = __shfl(dz, g - 1, LPT);
                            if(l >= g) add_exact(px, rx, ex), add_exact(py, ry, ey), add_exact(pz, rz, ez);
                        }
                    rx = known(rx), ry = known(ry), rz = known(rz);
                    const float qx = px + (rx + dx), qy = py + (ry + dy), qz = pz + (rz + dz);  // x_{t+1}
                    add_exact(px, rx, dx), add_exact(py, ry, dy), add_exact(pz, rz, dz);
                    px = __shfl(px, LPT - 1, LPT), py = __shfl(py, LPT - 1, LPT), pz = __shfl(pz, LPT - 1, LPT);
                    rx = __shfl(rx, LPT - 1, LPT), ry = __shfl(ry, LPT - 1, LPT), rz = __shfl(rz, LPT - 1, LPT);
                    // boxes s, s + 4, ... against this lane's step, each read
                    // while the one before it is worked on
                    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, flat = 0.0f;
                    const bool plain = scenePlain | !(fmaxf(fmaxf(fabsf(qx), fabsf(qy)), fabsf(qz)) < INFINITY) |
                                       __builtin_isunordered(qx, qy) | (qz != qz);
                    const uint64_t anyPlain = __builtin_amdgcn_ballot_w64(plain);
                    float4 lo = sBox[s], hi = sBox[nBox + s];
                    for(uint32_t o = s; o < nObs; o += 4)
                        {
                            const float4 l1 = sBox[o + 4], h1 = sBox[nBox + o + 4];
                            box_penalty(lo, hi, qx, qy, qz, ap.margin, ap.tau, K, plain, anyPlain, acc, flat);
                            lo = l1, hi = h1;
                        }
                    acc[0] += acc[0] + flat;
                    const float mine = ap.w_obstacle * quad_scatter(acc, l);
                    if(on)
                        {
                            const float Jt = (s == 0 ? mine : 0.0f) + ap.w_effort * d * d;
#pragma unroll
                            for(int k = 0; k < 64 / LPT; ++k)
                                if(k == ((t0 / CH) & (64 / LPT - 1))) Jp[k] += Jt;
                            Wg[(size_t)t * 8 + s] = mine;
                        }
                }
#pragma unroll
            for(int k = 0; k < 64 / LPT; ++k)
                {
#pragma unroll
                    for(int o = 1; o < LPT; o <<= 1) Jp[k] += __shfl_xor(Jp[k], o, 64);
                }
            float J = Jp[0];
            if(LPT == 32) J = J + Jp[64 / LPT - 1];
            if(LPT == 16) J = (J + Jp[1 % (64 / LPT)]) + (Jp[2 % (64 / LPT)] + Jp[64 / LPT - 1]);
            const float ex = (px - gx) + known(rx), ey = (py - gy) + known(ry), ez = (pz - gz) + known(rz);
            J += ap.w_goal * (ex * ex + ey * ey + ez * ez);
            if(act && l == 0) cost[(size_t)it * N + i] = J;
            if(REFINE)
                {
                    if(it == iters) break;
                    b1t *= ap.beta1;
                    b2t *= ap.beta2;
                }
            __threadfence_block();  // the penalty gradients
            // 3. backward, the last round first. lam: adjoint j of the chain;
            // lx, ly, lz, l5: adjoints of the position and of psi at the end
            // of the round
            float lam = 0.0f, l5 = 0.0f;
            float lx = 2.0f * ap.w_goal * ex, ly = 2.0f * ap.w_goal * ey, lz = 2.0f * ap.w_goal * ez;
            float4 wn, gn;
            float un = 0.0f, mn = 0.0f, qn = 0.0f;
            auto fetch3 = [&](int t) {
                const int tc     = t < 0 ? 0 : t < tl ? t : tl;
                const float4* w4 = reinterpret_cast<const float4*>(W + (size_t)tc * kStageWords);
                an = w4[s], vn = w4[4 + s], wn = w4[8 + s];
                gn = *reinterpret_cast<const float4*>(Wg + (size_t)tc * 8);
                un = Wg[(size_t)tc * 8 + 4 + s];
                if(REFINE && it > 0) mn = Wm[(size_t)tc * 8 + s], qn = Wm[(size_t)tc * 8 + 4 + s];
            };
            const int last = (Tm - 1) / CH * CH;
            if(Tm > 0) fetch3(last + tt);
            for(int t0 = last; t0 >= 0 && Tm > 0; t0 -= CH)
                {
                    const int t     = t0 + tt;
                    const bool on   = t < T;
                    const float4 a = an, v4 = vn, w = wn, g4 = gn;
                    const float uc = un;
                    float mom = mn, vel = qn;
                    fetch3(t - CH);
                    float sf, cf, st, ct, sp, cp;
                    sincos_fused(a.x, sf, cf);
                    sincos_fused(a.y, st, ct);
                    sincos_fused(a.z, sp, cp);
                    // adjoint of x_{t+1}'s position: gradients at x_{t+1} .. x_T
                    float hx = on ? g4.y : 0.0f, hy = on ? g4.z : 0.0f, hz = on ? g4.w : 0.0f;
#pragma unroll
                    for(int o = 4; o < 16; o <<= 1)
                        {
                            const float fx = __shfl_down(hx, o, 16), fy = __shfl_down(hy, o, 16);
                            const float fz = __shfl_down(hz, o, 16);
                            if((l & 15) + o < 16) hx += fx, hy += fy, hz += fz;
                        }
#pragma unroll
                    for(int g = LPT - 16; g > 0; g -= 16)
                        {
                            const float fx = __shfl(hx, g, LPT), fy = __shfl(hy, g, LPT), fz = __shfl(hz, g, LPT);
                            if(l < g) lx += fx, ly += fy, lz += fz;
                        }
                    hx += lx, hy += ly, hz += lz;
                    lx = __shfl(hx, 0, LPT), ly = __shfl(hy, 0, LPT), lz = __shfl(hz, 0, LPT);
                    const float a0 = hS * hx, a1 = hS * hy, a2 = hS * hz;
                    const float U = v4.x, V = v4.y, Wv = v4.z, p = w.x, q = w.y, r = w.z;
                    const float R00 = ct * cp, R01 = sf * st * cp - cf * sp, R02 = cf * st * cp + sf * sp;
                    const float R10 = ct * sp, R11 = sf * st * sp + cf * cp, R12 = cf * st * sp - sf * cp;
                    const float R21 = sf * ct, R22 = cf * ct;
                    const float m  = sf * V + cf * Wv, be = cf * V - sf * Wv;
                    const float al = ct * U + st * m, rt = ct * m - st * U;
                    // adjoint of psi (the derivative of the world velocity by psi)
                    const float g5 = (cp * al - sp * be) * a1 - (sp * al + cp * be) * a0;
                    float h5       = quad_sum(g5);
                    h5             = on ? h5 : 0.0f;
#pragma unroll
                    for(int o = 4; o < 16; o <<= 1)
                        {
                            const float f5 = __shfl_down(h5, o, 16);
                            if((l & 15) + o < 16) h5 += f5;
                        }
#pragma unroll
                    for(int g = LPT - 16; g > 0; g -= 16)
                        {
                            const float f5 = __shfl(h5, g, LPT);
                            if(l < g) l5 += f5;
                        }
                    const float n5 = __shfl_down(h5, 4, 16);
                    const float m5 = l5 + ((l & 15) + 4 < 16 ? n5 : 0.0f);  // of x_{t+1}
                    l5 = __shfl(l5 + h5, 0, LPT);
                    const float hG = s == 3 ? 0.0f : s == 2 ? K.h : K.hh;
                    const float a5 = hS * m5 + hG * dpp<0xF9>(g5);  // quad_perm [1,2,3,3]: the stage after
                    // the stage's rows
                    const float ict = recip(ct), tn = st * ict;
                    const float E = q * sf + r * cf, F = q * cf - r * sf;
                    const float nv = __builtin_amdgcn_sqrtf(U * U + V * V + Wv * Wv);
                    const float nw = __builtin_amdgcn_sqrtf(p * p + q * q + r * r);
                    const float mN = -K.minv * K.nu * nv, kv = nv > 0.0f ? -K.minv * K.nu * recip(nv) : 0.0f;
                    const float M  = -K.mu * nw, km = nw > 0.0f ? -K.mu * recip(nw) : 0.0f;
                    const float kU = kv * U, kV = kv * V, kW = kv * Wv, kp = km * p, kq = km * q, kr = km * r;
                    const float gct = K.g * ct, gst = K.g * st;
                    const float d0f = R02 * V - R01 * Wv, d1f = R12 * V - R11 * Wv, d2f = R22 * V - R21 * Wv;
                    const float d0t = cp * rt, d1t = sp * rt, d2t = -al;
                    float* B        = L.coef + lane * kBlockWords;
                    auto row = [&](int k, float c, float x3, float x4, float x6, float x7, float x8, float x9,
                                   float x10, float x11) {
                        float4* o = reinterpret_cast<float4*>(B + k * kRowWords);
                        o[0] = make_float4(c, x3, x4, x6);
                        o[1] = make_float4(x7, x8, x9, x10);
                        B[k * kRowWords + 8] = x11;
                    };
                    row(0, d0f * a0 + d1f * a1 + d2f * a2 + F * ict * a5, F * tn, -E, 0.0f, gct * cf, -gct * sf, 0.0f,
                        0.0f, 0.0f);
                    row(1, d0t * a0 + d1t * a1 + d2t * a2 + E * tn * ict * a5, E * ict * ict, 0.0f, -gct, -gst * sf,
                        -gst * cf, 0.0f, 0.0f, 0.0f);
                    row(2, R00 * a0 + R10 * a1 - st * a2, 0.0f, 0.0f, mN + kU * U, kU * V - r, kU * Wv + q, 0.0f, 0.0f,
                        0.0f);
                    row(3, R01 * a0 + R11 * a1 + R21 * a2, 0.0f, 0.0f, kU * V + r, mN + kV * V, kV * Wv - p, 0.0f, 0.0f,
                        0.0f);
                    row(4, R02 * a0 + R12 * a1 + R22 * a2, 0.0f, 0.0f, kU * Wv - q, kV * Wv + p, mN + kW * Wv, 0.0f,
                        0.0f, 0.0f);
                    row(5, 0.0f, 1.0f, 0.0f, 0.0f, Wv, -V, K.bx * (M + kp * p), K.ay * r + K.by * kp * q,
                        K.az * q + K.bz * kp * r);
                    row(6, sf * ict * a5, sf * tn, cf, -Wv, 0.0f, U, K.ax * r + K.bx * kq * p, K.by * (M + kq * q),
                        K.az * p + K.bz * kq * r);
                    row(7, cf * ict * a5, cf * tn, -sf, V, -U, 0.0f, K.ax * q + K.bx * kr * p, K.ay * p + K.by * kr * q,
                        K.bz * (M + kr * r));
                    wave_sync();
                    // the chain over this round's steps
                    for(int k = (Tm - 1 - t0 < CH - 1 ? Tm - 1 - t0 : CH - 1); k >= 0; --k)
                        {
                            const float* B0 = L.coef + (gb + 4 * k) * kBlockWords + j * kRowWords;
                            auto apply = [&](int stage, float x) {
                                const float* b   = B0 + stage * kBlockWords;
                                const float4 c0 = *reinterpret_cast<const float4*>(b);
                                const float4 c1 = *reinterpret_cast<const float4*>(b + 4);
                                const float c8  = b[8];
                                float y         = c0.x;
                                row_madd(y, x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w, c8);
                                return y;
                            };
                            float x = K.h6 * lam, sum = x;
                            float y = apply(3, x), xb = lam + y;
                            x = K.h3 * lam + K.h * y, sum += x;
                            y = apply(2, x), xb += y;
                            x = K.h3 * lam + K.hh * y, sum += x;
                            y = apply(1, x), xb += y;
                            x = K.h6 * lam + K.hh * y, sum += x;
                            y = apply(0, x), xb += y;
                            lam = t0 + k < T ? xb : lam;
                            // rows 4..7 (a8 .. a11): the adjoints of controls 0..3, unscaled
                            if(j >= 4) L.ubar[gb + 4 * k + j - 4] = sum;
                        }
                    wave_sync();
                    const float gk = uscale * L.ubar[lane] + 2.0f * ap.w_effort * (uc - uref);
                    const size_t iu = ((size_t)t * 4 + s) * N + i;
                    if(on)
                        {
                            if(REFINE)
                                {
                                    mom = ap.beta1 * mom + (1.0f - ap.beta1) * gk;
                                    vel = ap.beta2 * vel + (1.0f - ap.beta2) * gk * gk;
                                    Wm[(size_t)t * 8 + s]     = mom;
                                    Wm[(size_t)t * 8 + 4 + s] = vel;
                                    float u1 = uc - ap.lr * (mom / (1.0f - b1t)) /
                                                      (__builtin_sqrtf(vel / (1.0f - b2t)) + ap.adam_eps);
                                    if(ap.clamp) u1 = u1 < umin ? umin : (u1 > umax ? umax : u1);
                                    u[iu]                     = u1;
                                    Wg[(size_t)t * 8 + 4 + s] = u1;
                                }
                            else
                                grad[iu] = gk;
                        }
                    wave_sync();  // the next round rewrites the rows
                }
            if(REFINE) __threadfence_block();  // the controls, read by other lanes in the next pass
        }
    if(!REFINE && act)
        for(uint32_t t = (uint32_t)T + tt; t < maxT; t += CH) grad[((size_t)t * 4 + s) * N + i] = 0.0f;
}

// floats of `work` per trajectory
static size_t rollout_words(bool refine, uint32_t maxT)
{
    return (size_t)maxT * (kStageWords + 8 + (refine ? 8 : 0));
}

// lanes per trajectory: all 64 while the waves fit the chip's SIMDs one each
// (more lanes share the boxes and the steps of a round; the chains do not get
// shorter), fewer above
static uint32_t rollout_lanes(uint32_t n)
{
    return n <= 1024 ? 64 : n <= 2048 ? 32 : 16;
}

// Trajectories per launch, and the floats of work space they take. The launches
// of a call share one work space: 1 GiB, or, of long rollouts, 12 floats a step
// and trajectory (20 with moments) where that is more: a launch lasts as long
// as the longest chain, however few trajectories it holds, so at most five
// launches do the call (4096 trajectories of 8000 and 20000 steps: 74 and 484 ms
// in launches of 1 GiB, 47 and 117 in five; 77 and 193 in one launch of a kernel
// that kept 12 floats a step and ran the whole step in every lane).
uint32_t rollout_slab(bool refine, uint32_t n, uint32_t maxT, size_t* floats)
{
    const size_t per  = std::max<size_t>(rollout_words(refine, maxT), 1);
    const size_t most = std::max<size_t>(size_t(1) << 28, ((size_t)maxT * (refine ? 20 : 12) + 12) * n) / per;
    const size_t wave = 64 / rollout_lanes(n), all = ((size_t)n + wave - 1) / wave * wave;
    // whole waves: four trajectories at most
    const size_t slab = most >= all ? all : most >= 4 ? most / 4 * 4 : std::max<size_t>(most, 1);
    *floats = per * slab;
    return (uint32_t)slab;
}

template <bool REFINE, int LPT>
static void launch_rollout_lanes(const RolloutK& K, const kgmt_adjoint_params& ap, uint32_t i0, uint32_t cnt,
                                 uint32_t n, uint32_t maxT, const int32_t* steps, const float* x0, const float* goal,
                                 float* u, float* grad, float* work, const float* rows, uint32_t nObs, float* cost,
                                 hipStream_t s)
{
    const dim3 g((cnt + 64 / LPT - 1) / (64 / LPT)), b(64);
    const size_t lds = (size_t)box_slots(nObs) * 2 * sizeof(float4);
    hipLaunchKernelGGL((k_rollout<REFINE, LPT>), g, b, lds, s, K, ap, i0, n, maxT, steps, x0, goal, u, grad, work, rows,
                       nObs, cost);
}

hipError_t launch_rollout(bool refine, const RolloutK& K, const kgmt_adjoint_params& ap, uint32_t n, uint32_t maxT,
                          const int32_t* steps, const float* x0, const float* goal, float* u, float* grad, float* work,
                          uint32_t slab, const float* rows, uint32_t nObs, float* cost, hipStream_t s)
{
    for(uint32_t i0 = 0; i0 < n; i0 += std::min(slab, n - i0))
        {
            const uint32_t cnt = std::min(slab, n - i0);
            auto go            = [&](auto kernel) { kernel(K, ap, i0, cnt, n, maxT, steps, x0, goal, u, grad, work, rows, nObs, cost, s); };
            switch(rollout_lanes(cnt))
                {
                    case 64: refine ? go(launch_rollout_lanes<true, 64>) : go(launch_rollout_lanes<false, 64>); break;
                    case 32: refine ? go(launch_rollout_lanes<true, 32>) : go(launch_rollout_lanes<false, 32>); break;
                    default: refine ? go(launch_rollout_lanes<true, 16>) : go(launch_rollout_lanes<false, 16>); break;
                }
            const hipError_t e = hipGetLastError();
            if(e != hipSuccess) return e;
        }
    return hipSuccess;
}

}  // namespace kgmt
