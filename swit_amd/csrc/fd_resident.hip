// Resident time loops: the wavefields of a shot stay in registers for the whole loop.
//
// The step kernels of fd_batched.hip read and write every field once per time step, so a
// step cannot be faster than HBM (219.8 MB a forward step at 481x141 with 49 shots, 37 us
// at the 5.9 TB/s that plain streaming reaches; the kernel took 38.8 us).  The state itself
// is small: 73 MB there, against 128 MB of vector registers on the chip.  Here one launch
// runs many time steps.  A shot is cut into P windows of columns, one workgroup each, which
// hold p, u, w of their columns in registers; only the columns next to a window's edge are
// exchanged, through memory, and only receivers and boundary strips are written.
//
// Layout.  A lane holds R consecutive rows (rows z0 + lane R + r, so one wave spans the
// whole height: 64 R rows) of C consecutive columns; wave w of a workgroup holds columns
// w C .. w C + C - 1 of the window.  Stencils along z stay inside the lane except at its
// first and last rows, which the neighbouring lanes hand over by wave shifts; stencils
// along x stay inside the thread except at the wave's first and last columns, which go
// through LDS (2 columns of p one way and 1 the other, the same for u).  A step is then
// two phases (p, then u and w) with one barrier each.
//
// Windows overlap: one reaches 3 columns past its own columns on each inner side.  p needs u
// at x-2..x+1 and u needs p at x-1..x+2, so with fresh u in the 3 columns after every forward
// step (fresh p after every reverse step) the rest of the halo that is needed keeps itself
// right.  The columns that are sent and received always are the first and last six of a
// window, so they sit in known registers of its first and last waves.  These run the step's
// second phase at raised priority, send, and wait for the neighbour while the other waves
// still compute.  A message word is 8 bytes, {value, number
// of the message}, stored and polled with relaxed agent-scope atomics: the word that carries
// a value also says that it has arrived, so no flag, fence or cache flush is needed (measured
// between workgroups on different XCDs, 64 words: 0.93 us per exchange with tagged words,
// 2.7 us and more with data, fence and flag).  Two slots alternate: a neighbour sends message
// n+2 only after it has received n+1, which is sent after n was read.
//
// Progress.  Workgroups take their place by a ticket counter when they start to run, and P
// consecutive tickets form the group of one shot.  So at any time at most one group of a
// launch is incomplete, and it waits only for workgroups that are dispatched next; complete
// groups run to their end.  Several such launches at once hold at most P - 1 waiting
// workgroups each, P at most a quarter of the chip's places, so with up to four at once (the
// hardware queues of a process) one of them always completes.  Every wait is bounded by the
// clock all the same (fd_wait.h): past that a wave stops waiting for good, sets Ctl::err, and
// the job's outputs are overwritten with NaN.  What an unfinished forward saved for an adjoint
// stays marked (Ctl::bad), over other jobs and for the step kernels too, until a forward that
// finishes takes its place: the adjoints' outputs are NaN as well.
//
// Per-cell arithmetic and its order are those of the step kernels: results are the same
// bits.  Cells outside an update region have K (or B) = 0 and hold zeros, so they need no
// test: fac * 0 - 0 * d = 0.
#include "fd_common.h"
#include "fd_kernels.h"
#include "fd_wait.h"

namespace swit {
namespace rk {

typedef unsigned long long u64;


// lane l gets lane l+1's (up) or l-1's (dn) value, 0 past the ends; every lane active
__device__ __forceinline__ float up1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ float dn1(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}

// Barrier for LDS alone: __syncthreads also waits for every global store in flight, and
// with it for the acknowledgement of message words, receiver samples and strips.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One window configuration.
struct Cfg {
    int R, C, W, P;      // rows per lane, columns per wave, waves, windows per shot
    int G;               // groups (shots in flight)
    int z0;              // padded row of lane 0's first row
};
constexpr int kH = 3;    // halo columns
// Columns: window j covers W C columns from 1 + j (W C - 2 kH).
__host__ __device__ inline int window_x(int W, int C, int j) { return 1 + j * (W * C - 2 * kH); }
__host__ __device__ inline int window_os(int W, int C, int j) { return window_x(W, C, j) + (j > 0 ? kH : 0); }
__host__ __device__ inline int window_oe(int W, int C, int j, int P, int nxp) {
    return j + 1 < P ? window_x(W, C, j) + W * C - 1 - kH : nxp;
}

constexpr int kHistPad = 64 * 8;    // floats past the divergence history: a column's lanes past the grid read them

// What a forward saves for an adjoint: strips and final state, or the exact forward's history.
enum Saved { kNothing = -1, kStrips = 0, kHistory = 1 };

struct Ctl {
    unsigned ticket;
    int err;                 // a wait of the job under way ran out
    int bad[2];              // the saved strips, history are an unfinished forward's
};

struct FwdArgs {
    Dims d;
    Cfg c;
    int s0, ns;                 // shots s0 .. s0 + ns - 1
    int it0, it1;               // steps it0 .. it1
    const float *co;            // [1 + ncol][5][64 R] coefficients of columns 0 .. ncol (k_res_setup)
    int ncol;
    const float *fpx;           // [1 + ncol] 1 - kappa_p of a column's own layer
    const ShotGeom *geo;
    const float *src;           // [ns][nt]
    // Receivers.  Staged (most surveys: few distinct rows): a window's receivers leave through
    // the p stage; rtab [ns][P][2][W * 64]: stage offset of a receiver, -1 none, rbase [ns][P]:
    // first slot.  Direct (rtab null): rec [ns][P][W * 64] {cells of the thread with a
    // receiver (64 bits), first slot, 0}.
    const int *rtab, *rbase;
    const uint4 *rec;
    unsigned long long pmask;   // lanes whose p rows are staged (strip rows, receiver rows)
    float *seis_t;              // [ns][nt][ngmax], receivers in slot order
    float *strips;              // null, or [ns][s_rows][S]: row (it - 1) % s_rows
    int s_rows;
    DSave hist;
    const float *in;            // null (zero state) or [ns][3][nxp][ld]
    float *out;                 // null or [ns][3][nxp][ld]
    float *end;                 // null or [ns][3][nx][nz]
    u64 *msg;                   // [G P][2 slots][2 sides][3 R][64]
    Ctl *ctl;
    unsigned limit;             // of a wait (wait_limit)
};

// A value the compiler must take as changed: what is computed or loaded from it inside a
// time step stays there instead of being carried (spilled) across the whole time loop.
__device__ __forceinline__ void opaque_s(int &v) {
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
}
__device__ __forceinline__ void opaque_v(unsigned &v) { asm volatile("" : "+v"(v)); }
// The value is computed by here: the compiler may not move its arithmetic further down.
__device__ __forceinline__ void pin(float &v) { asm volatile("" : "+v"(v)); }

// The kernel's arguments as they lie in memory.  Taken anew (opaque) where a step needs one
// that is not used all the time, so that it is loaded there instead of being held, or
// spilled to vector lanes, over the whole loop.
template <class A> using ArgPtr = const __attribute__((address_space(4))) A *;
template <class A> __device__ __forceinline__ ArgPtr<A> fresh_args() {
    ArgPtr<A> k = (ArgPtr<A>)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return k;
}

// A workgroup's place: its ticket, and the ticket behind its group's last.
__device__ __forceinline__ void take_place(Ctl *ctl, int P, unsigned (&place)[2]) {
    const unsigned t = atomicAdd(&ctl->ticket, 1u);
    place[0] = t;
    place[1] = (t / P + 1) * P;
}

// One column's rows into a message (row r at o + 64 r words).
template <int R> __device__ __forceinline__ void send_col(u64 *o, unsigned tag, const float (&v)[R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        // through a register of its own: a word formed from the state's register would turn
        // that register into a pair for the whole time loop
        unsigned b;
        asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(v[r]));
        __hip_atomic_store(o + r * 64, ((u64)tag << 32) | b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
// N columns' rows out of a message, polled until every word carries the tag (all loads of a
// round in flight together).  A wave that has waited too long once waits no more.  The group is
// looked at past the first limit only: a look at every start of a launch took 2 us of it.  The
// limit is read where a poll has failed: taken before the polls, a step of the exact
// forward of 76 shots of 472x179 took 28.9 us (28.0).
template <class A, int R, int N>
__device__ __forceinline__ void recv_cols(const u64 *in, unsigned tag, const unsigned (&place)[2], bool &dead,
                                          float (&v)[N][R]) {
    u64 from = 0, q[N][R];
    for (;;) {
        unsigned bad = 0;
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                q[n][r] = __hip_atomic_load(in + (n * R + r) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                bad |= (unsigned)(q[n][r] >> 32) ^ tag;
            }
        if (__all(bad == 0) || dead) break;
        const ArgPtr<A> k = fresh_args<A>();
        const u64 now = wall_clock64();
        const unsigned limit = k->limit;
        Ctl *ctl = k->ctl;
        if (wait_over(now, from, limit) &&
            (__hip_atomic_load(&ctl->ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= place[1] ||
             wait_over(now, from, kRoomWaits * limit))) {
            dead = true;
            if ((threadIdx.x & 63) == 0) __hip_atomic_store(&ctl->err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
    }
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int r = 0; r < R; ++r)      // as in send_col
            asm volatile("v_mov_b32 %0, %1" : "=v"(v[n][r]) : "v"((unsigned)q[n][r]));
}

// A window's first and last six columns: position q from the left (right) end lies in wave
// q / C (W - 1 - q / C) at column q % C (C - 1 - q % C).  Sends the three own columns next to
// each neighbour (positions 3, 4, 5) into its inbox; halo column h of the left window's right
// side is this window's position 3 + h, of the right window's left side position 5 - h.
template <int R, int C>
__device__ __forceinline__ void send_edges(bool has_l, bool has_r, int wave, int W, u64 *to_l, u64 *to_r, unsigned tag,
                                           const float (&f)[C][R]) {
#pragma unroll
    for (int h = 0; h < kH; ++h) {
        const int ql = kH + h, qr = 2 * kH - 1 - h;
        if (has_l && wave == ql / C) send_col<R>(to_l + h * R * 64, tag, f[ql % C]);
        if (has_r && wave == W - 1 - qr / C) send_col<R>(to_r + h * R * 64, tag, f[C - 1 - qr % C]);
    }
}
// Fresh halo columns from the inboxes: positions 0, 1, 2 from each end (C >= 3: one wave).
template <class A, int R, int C>
__device__ __forceinline__ void recv_edges(bool has_l, bool has_r, int wave, int W, const u64 *from_l,
                                           const u64 *from_r, unsigned tag, const unsigned (&place)[2],
                                           bool &dead, float (&f)[C][R]) {
    float v[kH][R];
    if (has_l && wave == 0) {
        recv_cols<A, R, kH>(from_l, tag, place, dead, v);
#pragma unroll
        for (int h = 0; h < kH; ++h)
#pragma unroll
            for (int r = 0; r < R; ++r) f[h][r] = v[h][r];
    }
    if (has_r && wave == W - 1) {
        recv_cols<A, R, kH>(from_r, tag, place, dead, v);
#pragma unroll
        for (int h = 0; h < kH; ++h)
#pragma unroll
            for (int r = 0; r < R; ++r) f[C - kH + h][r] = v[h][r];
    }
}

// LDS of a workgroup: the waves' edge columns, the p stage (NS lanes), the u, w stage.
__host__ __device__ inline int lds_edge_floats(int W, int R) { return W * 6 * R * 64; }
__host__ __device__ inline int lds_stage_floats(int W, int C, int R, int NS) { return W * C * (NS + 8) * R; }

// R consecutive floats from a buffer: byte offset voff of this lane plus the wave-uniform soff
typedef unsigned vec2 __attribute__((ext_vector_type(2)));
typedef unsigned vec3 __attribute__((ext_vector_type(3)));
typedef unsigned vec4 __attribute__((ext_vector_type(4)));
template <int R>
__device__ __forceinline__ void buffer_rows(__amdgpu_buffer_rsrc_t rs, unsigned voff, int soff, float (&v)[R]) {
    constexpr int N = R >= 4 ? 4 : R;
    if constexpr (N == 4) {
        const vec4 q = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, 0);
        for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(q[i]);
    } else if constexpr (N == 3) {
        const vec3 q = __builtin_amdgcn_raw_buffer_load_b96(rs, voff, soff, 0);
        for (int i = 0; i < 3; ++i) v[i] = __uint_as_float(q[i]);
    } else if constexpr (N == 2) {
        const vec2 q = __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0);
        for (int i = 0; i < 2; ++i) v[i] = __uint_as_float(q[i]);
    }
    if constexpr (R > 4) {
        constexpr int M = R - 4;
        if constexpr (M == 1) {
            v[4] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, voff + 16, soff, 0));
        } else if constexpr (M == 2) {
            const vec2 q = __builtin_amdgcn_raw_buffer_load_b64(rs, voff + 16, soff, 0);
            for (int i = 0; i < 2; ++i) v[4 + i] = __uint_as_float(q[i]);
        } else if constexpr (M == 3) {
            const vec3 q = __builtin_amdgcn_raw_buffer_load_b96(rs, voff + 16, soff, 0);
            for (int i = 0; i < 3; ++i) v[4 + i] = __uint_as_float(q[i]);
        } else {
            const vec4 q = __builtin_amdgcn_raw_buffer_load_b128(rs, voff + 16, soff, 0);
            for (int i = 0; i < 4; ++i) v[4 + i] = __uint_as_float(q[i]);
        }
    }
}
template <int R>
__device__ __forceinline__ void buffer_store_rows(__amdgpu_buffer_rsrc_t rs, unsigned voff, int soff,
                                                  const float (&v)[R]) {
    auto bits = [&](int i) { return __float_as_uint(v[i]); };
    if constexpr (R == 2) {
        __builtin_amdgcn_raw_buffer_store_b64(vec2{bits(0), bits(1)}, rs, voff, soff, 0);
    } else if constexpr (R == 3) {
        __builtin_amdgcn_raw_buffer_store_b96(vec3{bits(0), bits(1), bits(2)}, rs, voff, soff, 0);
    } else {
        __builtin_amdgcn_raw_buffer_store_b128(vec4{bits(0), bits(1), bits(2), bits(3)}, rs, voff, soff, 0);
        if constexpr (R == 5) __builtin_amdgcn_raw_buffer_store_b32(bits(R > 4 ? 4 : 0), rs, voff + 16, soff, 0);
        else if constexpr (R == 6)
            __builtin_amdgcn_raw_buffer_store_b64(vec2{bits(R > 4 ? 4 : 0), bits(R > 5 ? 5 : 0)}, rs, voff + 16, soff, 0);
        else if constexpr (R == 7)
            __builtin_amdgcn_raw_buffer_store_b96(vec3{bits(R > 4 ? 4 : 0), bits(R > 5 ? 5 : 0), bits(R > 6 ? 6 : 0)}, rs,
                                                  voff + 16, soff, 0);
        else if constexpr (R == 8)
            __builtin_amdgcn_raw_buffer_store_b128(vec4{bits(R > 4 ? 4 : 0), bits(R > 5 ? 5 : 0), bits(R > 6 ? 6 : 0),
                                                        bits(R > 7 ? 7 : 0)}, rs, voff + 16, soff, 0);
    }
}

// After buffer_store_rows of a, b, c: their registers stand until the stores have read them.  A vector
// instruction right behind a store of more than 64 bits may overwrite the store's last registers
// first; the compiler keeps two wait states clear only where the store's offset is no scalar
// register.  Measured: with v_sub_f32 v8 behind buffer_store_dwordx3 v[6:8] (3 and 4 rows a lane), 100
// of 36000 values of the backward illumination of 8 shots of 300x120 were another register's.
template <int R> __device__ __forceinline__ void after_stores(const float (&a)[R], const float (&b)[R], const float (&c)[R]) {
    if constexpr (R > 2) {
        asm volatile("s_nop 1");
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : : "v"(a[r]), "v"(b[r]), "v"(c[r]));
    }
}

// Forward steps it0 .. it1 (fdcore.f90:75-160) of every shot, the state in registers.
// Bound by vector issue: 28 operations per cell and step without contraction (the
// reference's rounding), about 40 with shifts, receivers and exchange.  R C <= 20 (80 registers
// of state and K) runs at four waves per SIMD, above (up to 200) at two.
// HIST: also store the divergence history (the exact adjoint's forward).
template <int R, int C, bool HIST>
__global__ __launch_bounds__(R *C > 20 ? 512 : 1024) void k_fwd_resident(FwdArgs a) {
    extern __shared__ float lds[];
    __shared__ unsigned sh_place[2];
    constexpr int PF = R * C > 20 ? 2 : 1;               // columns whose coefficients are in flight
    constexpr int kCol = 64 * R * 4;                     // bytes of a column of one array
    const int W = a.c.W, P = a.c.P;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) take_place(a.ctl, P, sh_place);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(sh_place[0]);
    const int grp = __builtin_amdgcn_readfirstlane(t / P), j = __builtin_amdgcn_readfirstlane(t % P);
    float *eU = lds;                                     // [W][3][R][64]: first, last but one, last column of u
    float *eP = eU + W * 3 * R * 64;                     // [W][3][R][64]: first, second, last column of p
    const int NS = __popcll(a.pmask);
    float *sp = eP + W * 3 * R * 64;                     // p stage [NS][W C][R]
    float *sv = sp + W * C * NS * R;                     // u, w stage [2][4][W C][R]

    // this wave's first column; the first and the last waves exchange with the neighbours
    const int x0w = window_x(W, C, j) + wave * C;
    const bool has_l = j > 0, has_r = j + 1 < P;
    const bool edge = (has_l && wave <= (2 * kH - 1) / C) || (has_r && wave >= W - 1 - (2 * kH - 1) / C);
    const unsigned voff0 = lane * R * 4;                 // byte offset of this lane's rows in a column
    const bool mirror = a.d.free_surface == 1 && lane == 0;
    // any column in the side layers: their damping factors differ along x; the other waves
    // take one column's factors for all of theirs (column 0 of the coefficient array)
    const bool wave_pml = x0w <= a.d.npml || x0w + C - 1 >= a.d.npml + a.d.nx;
    const __amdgpu_buffer_rsrc_t co = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.co), 0, (int)((unsigned)(a.ncol + 1) * 5u * kCol), 0x00027000);
    unsigned tag = 0;
    bool dead = false;
    // The pressure phase loads nothing: K stays in registers, and 1 - kappa_p is the smaller
    // of the column's and the row's (the damping is the larger of the two layers' profiles,
    // and 1 - damp dt rounds monotonically).  So the stores at a step's end (loads wait for
    // every earlier store: the counter is in order) complete behind it.
    float K[C][R], fpz[R];
#pragma unroll
    for (int c = 0; c < C; ++c) buffer_rows<R>(co, voff0, (x0w + c) * (5 * kCol), K[c]);
    buffer_rows<R>(co, voff0, 2 * kCol, fpz);

    const bool p_lane = (a.pmask >> lane) & 1;
    const int p_slot = __popcll(a.pmask & ((1ull << lane) - 1));
    // strip values this thread copies from the stages: NP of p (5 per column), NV of u, w (4)
    constexpr int NP = (5 * C + 63) / 64, NV = (4 * C + 63) / 64;
    int sp_lds[NP], sp_slot[NP], sv_lds[NV], sv_slot[NV];
#pragma unroll
    for (int i = 0; i < NP; ++i) sp_lds[i] = -1;
#pragma unroll
    for (int i = 0; i < NV; ++i) sv_lds[i] = -1;
    bool v_lane = false;
    int v_slot = 0;
    if (a.strips) {
        const int npml = a.d.npml, nx = a.d.nx, nz = a.d.nz, xw = window_x(W, C, j);
        const int os = window_os(W, C, j), oe = window_oe(W, C, j, P, a.d.nxp);
        const int lb = (nz - 1 + npml - a.c.z0) / R;     // lane of interior row nz - 1
        v_lane = lane < 2 || lane == lb || lane == lb + 1;
        v_slot = lane < 2 ? lane : 2 + lane - lb;
        const int top0 = 3 * nx + 6 * nz;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int n = threadIdx.x + i * W * 64, col = n / 5, v = n % 5, x = xw + col, jx = x - npml;
            if (col < W * C && x >= os && x <= oe && jx >= 1 && jx <= nx) {
                const int jz = v < 3 ? v + 1 : v == 3 ? nz : nz - 1;
                const int q = jz + npml - a.c.z0, L = q / R;
                sp_lds[i] = (__popcll(a.pmask & ((1ull << L) - 1)) * W * C + col) * R + q % R;
                sp_slot[i] = v < 3 ? top0 + 6 * (jx - 1) + v : 3 * (jx - 1) + v - 3;
            }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int n = threadIdx.x + i * W * 64, col = n / 4, v = n % 4, x = xw + col, jx = x - npml;
            if (col < W * C && x >= os && x <= oe && jx >= 1 && jx <= nx) {
                // u of rows 1 and 2, w of row 1, w of row nz - 1
                const int jz = v < 2 ? v + 1 : v == 2 ? 1 : nz - 1;
                const int q = jz + npml - a.c.z0, L = q / R;
                sv_lds[i] = (((v < 2 ? 0 : 4) + (L < 2 ? L : 2 + L - lb)) * W * C + col) * R + q % R;
                sv_slot[i] = v < 3 ? top0 + 6 * (jx - 1) + 3 + v : 3 * (jx - 1) + 2;
            }
        }
    }
    // one side column of the strips (interior columns 1, 2, nx - 1, nx): its rows of field
    // column `v` to row[3 nx + 6 (jz - 1) + q]
    auto side_column = [&](ArgPtr<FwdArgs> k, float *row, int x, unsigned voff, int q, const float (&v)[R]) {
        if (q < 0 || x < window_os(k->c.W, C, j) || x > window_oe(k->c.W, C, j, k->c.P, k->d.nxp)) return;
        const int jz0 = k->c.z0 + (int)(voff >> 2) - k->d.npml, nz = k->d.nz;
        float *o = row + 3 * k->d.nx + q;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (jz0 + r >= 1 && jz0 + r <= nz) o[6 * (jz0 + r - 1)] = v[r];
    };
    auto copy_velocities = [&](ArgPtr<FwdArgs> k, int s, int row) {
        float *q = k->strips + ((size_t)s * k->s_rows + row % k->s_rows) * k->d.S;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (sv_lds[i] >= 0) q[sv_slot[i]] = sv[sv_lds[i]];
    };

    // HIST: a column's divergence terms of step it.  Few cells a thread (kLate): all of them at the
    // step's end, where nothing is loaded until they have arrived behind the next pressure phase;
    // more would not fit the registers, and go out as they are made, which the velocity
    // coefficients then wait for (loads complete after every earlier store).  161x61, 8 shots:
    // 2.84 us a step stored at once, 2.52 us late.
    constexpr bool kLate = HIST && R * C <= 12;
    auto store_hist = [&](int s, int it, int x, unsigned voff, const float (&dv)[R]) {
        const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
        const int zr = k->c.z0 + (int)(voff >> 2), nzp = k->d.nzp;
        if (x < window_os(k->c.W, C, j) || x > window_oe(k->c.W, C, j, k->c.P, k->d.nxp)) return;
        float *h = k->hist.p + ((size_t)s * k->hist.slots + (it - 1 - k->hist.base)) * (k->d.nxp * k->d.ld) +
                   (size_t)(x - 1) * k->d.ld;
        const unsigned o = zr - 1;
        if (zr + R - 1 <= nzp) {
            __builtin_memcpy(h + o, dv, sizeof(float) * R);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (zr + r <= nzp) h[o + r] = dv[r];
        }
    };

    for (int s = a.s0 + grp; s < a.s0 + a.ns; s += a.c.G) {
        const int isx = a.geo[s].isx, isz = a.geo[s].isz;
        const float *src = a.src + (size_t)s * a.d.nt;
        float p[C][R], u[C][R], w[C][R];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int r = 0; r < R; ++r) p[c][r] = u[c][r] = w[c][r] = 0.0f;
        if (a.in) {
            const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            const int zr = k->c.z0 + (int)(voff >> 2), ld = k->d.ld, np = k->d.nxp * ld;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                if (x0 + c > k->d.nxp) continue;
                const float *f = k->in + (size_t)s * 3 * np + (size_t)(x0 + c - 1) * ld;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (zr + r > k->d.nzp) continue;
                    const unsigned o = zr + r - 1;
                    p[c][r] = f[o];
                    u[c][r] = f[np + o];
                    w[c][r] = f[2 * np + o];
                }
            }
        }
        // receivers: stage offsets of this thread's two, or (direct) its cells' bits
        int ro0 = -1, ro1 = -1, rbase = 0;
        uint4 rec0 = make_uint4(0, 0, 0, 0);
        unsigned wm0 = 0, wm1 = 0;                           // cells with a receiver in any lane
        if (a.rtab) {
            const int *q = a.rtab + ((size_t)s * P + j) * 2 * (W * 64) + threadIdx.x;
            ro0 = q[0];
            ro1 = q[W * 64];
            rbase = a.rbase[s * P + j];
        } else {
            rec0 = a.rec[((size_t)s * P + j) * (W * 64) + threadIdx.x];
            wm0 = rec0.x;
            wm1 = rec0.y;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                wm0 |= __shfl_xor(wm0, o);
                wm1 |= __shfl_xor(wm1, o);
            }
            wm0 = __builtin_amdgcn_readfirstlane(wm0);
            wm1 = __builtin_amdgcn_readfirstlane(wm1);
        }

        // u of the edge columns for the next step
        auto put_u = [&]() {
            float *e = eU + (size_t)wave * 3 * R * 64 + lane;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                e[r * 64] = u[0][r];
                e[(R + r) * 64] = u[C - 2][r];
                e[(2 * R + r) * 64] = u[C - 1][r];
            }
        };
        // velocity coefficients of column c, in flight PF columns ahead
        float cB[PF + 1][R], cfu[PF + 1][R], cfw[PF + 1][R];
        auto fetch_v = [&](int x, unsigned voff, int c) {
            const int f = wave_pml ? (x + c) * (5 * kCol) : 0;
            buffer_rows<R>(co, voff, (x + c) * (5 * kCol) + kCol, cB[c % (PF + 1)]);
            buffer_rows<R>(co, voff, f + 3 * kCol, cfu[c % (PF + 1)]);
            buffer_rows<R>(co, voff, f + 4 * kCol, cfw[c % (PF + 1)]);
        };
        put_u();
        lds_barrier();
        float srcv = a.d.dt * src[a.it0 - 1];
        const int it1 = a.it1;
        for (int it = a.it0; it <= it1; ++it) {
            const float src_next = it < it1 ? src[it] : 0.0f;
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            float hd[kLate ? C : 1][R];
            // ---- p: u of the neighbouring waves' columns x0-2, x0-1 and x0+C ----
            {
                const ArgPtr<float> fpx = (ArgPtr<float>)fresh_args<FwdArgs>()->fpx + x0;
                float ul2[R], ul1[R], ur1[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float *e = eU + lane;
                    ul2[r] = wave > 0 ? e[(((wave - 1) * 3 + 1) * R + r) * 64] : 0.0f;
                    ul1[r] = wave > 0 ? e[(((wave - 1) * 3 + 2) * R + r) * 64] : 0.0f;
                    ur1[r] = wave + 1 < W ? e[((wave + 1) * 3 * R + r) * 64] : 0.0f;
                }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const float fx = fpx[c];
                    const float wd1 = dn1(w[c][R - 1]), wd2 = dn1(w[c][R - 2]), wu = up1(w[c][0]);
                    float dv[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float um1 = c >= 1 ? u[c - (c >= 1)][r] : ul1[r];
                        const float um2 = c >= 2 ? u[c - (c >= 2 ? 2 : 0)][r] : c == 1 ? ul1[r] : ul2[r];
                        const float up = c + 1 < C ? u[c + (c + 1 < C)][r] : ur1[r];
                        const float wm1 = r >= 1 ? w[c][r - (r >= 1)] : wd1;
                        const float wm2 = r >= 2 ? w[c][r - (r >= 2 ? 2 : 0)] : r == 1 ? wd1 : wd2;
                        const float wp1 = r + 1 < R ? w[c][r + (r + 1 < R)] : wu;
                        dv[r] = div_term(u[c][r], um1, up, um2, w[c][r], wm1, wp1, wm2);
                        p[c][r] = fminf(fx, fpz[r]) * p[c][r] - K[c][r] * dv[r];
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) pin(p[c][r]);
                    if constexpr (HIST) {
                        if constexpr (kLate) {
#pragma unroll
                            for (int r = 0; r < R; ++r) {
                                hd[c][r] = dv[r];
                                pin(hd[c][r]);
                            }
                        } else {
                            store_hist(s, it, x0 + c, voff, dv);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int c = 0; c < PF; ++c) fetch_v(x0, voff, c);
            // source (fdcore.f90:88-89)
            if ((unsigned)(isx - x0) < (unsigned)C) {
                const int zr = fresh_args<FwdArgs>()->c.z0 + (int)(voff >> 2);
#pragma unroll
                for (int c = 0; c < C; ++c)
                    if (x0 + c == isx) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            if (zr + r == isz) p[c][r] = p[c][r] + srcv;
                    }
            }
            // p mirror: lane 0 holds rows fs-1, fs, fs+1 (fs+1 in lane 1 when R = 2)
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float pm = R > 2 ? p[c][R > 2 ? 2 : 0] : up1(p[c][0]);
                if (mirror) p[c][0] = -pm;
            }
            {
                float *e = eP + (size_t)wave * 3 * R * 64 + lane;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    e[r * 64] = p[0][r];
                    e[(R + r) * 64] = p[1][r];
                    e[(2 * R + r) * 64] = p[C - 1][r];
                }
            }
            // p of the staged rows (receivers, strips); the last step's u, w leave their stage
            if (p_lane) {
                float *q = sp + (p_slot * W + wave) * (C * R);
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int r = 0; r < R; ++r) q[c * R + r] = p[c][r];
            }
            if (a.strips && it > a.it0) copy_velocities(fresh_args<FwdArgs>(), s, it - 2);
            lds_barrier();
            // ---- u, w: p of the neighbouring waves' columns x0-1, x0+C, x0+C+1 ----
            if (edge) __builtin_amdgcn_s_setprio(3);
            {
                float pl1[R], pr1[R], pr2[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float *e = eP + lane;
                    pl1[r] = wave > 0 ? e[(((wave - 1) * 3 + 2) * R + r) * 64] : 0.0f;
                    pr1[r] = wave + 1 < W ? e[((wave + 1) * 3 * R + r) * 64] : 0.0f;
                    pr2[r] = wave + 1 < W ? e[(((wave + 1) * 3 + 1) * R + r) * 64] : 0.0f;
                }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if (c + PF < C) fetch_v(x0, voff, c + PF);
                    const float pd = dn1(p[c][R - 1]), pu0 = up1(p[c][0]), pu1 = up1(p[c][1]);
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float xm = c >= 1 ? p[c - (c >= 1)][r] : pl1[r];
                        const float xp = c + 1 < C ? p[c + (c + 1 < C)][r] : pr1[r];
                        const float xq = c + 2 < C ? p[c + (c + 2 < C ? 2 : 0)][r] : c + 2 == C ? pr1[r] : pr2[r];
                        const float zm = r >= 1 ? p[c][r - (r >= 1)] : pd;
                        const float zp = r + 1 < R ? p[c][r + (r + 1 < R)] : pu0;
                        const float zq = r + 2 < R ? p[c][r + (r + 2 < R ? 2 : 0)] : r + 2 == R ? pu0 : pu1;
                        const float b = cB[c % (PF + 1)][r];
                        u[c][r] = v_update_f(u[c][r], b, cfu[c % (PF + 1)][r], p[c][r], xp, xq, xm);
                        w[c][r] = v_update_f(w[c][r], b, cfw[c % (PF + 1)][r], p[c][r], zp, zq, zm);
                    }
                    if (mirror) w[c][0] = w[c][1];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        pin(u[c][r]);
                        pin(w[c][r]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // ---- exchange, out: inboxes [group][window][slot][side], side 0 from the left ----
            const bool exch = it < it1;
            if (exch) ++tag;
            u64 *box = nullptr;
            constexpr int kMsg = kH * R * 64;
            if (edge && exch) {
                const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
                box = k->msg + ((size_t)(grp * k->c.P + j) * 2 + (tag & 1)) * (2 * kMsg) + voff / (4 * R);
                send_edges<R, C>(has_l, has_r, wave, W, box - 3 * kMsg, box + 4 * kMsg, tag, u);
            }
            // ---- receivers (fdcore.f90:123-128) and strips (:130-159): all stores of the step
            // come here, p stands since the pressure phase ----
            {
                const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
                float *q = k->seis_t + ((size_t)s * k->d.nt + (it - 1)) * k->d.ngmax + rbase;
                const int T = k->c.W * 64;
                if (ro0 >= 0) q[threadIdx.x] = sp[ro0];
                if (ro1 >= 0) q[threadIdx.x + T] = sp[ro1];
            }
            if (wm0 | wm1) {
                const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
                int m0 = __builtin_amdgcn_readfirstlane(wm0), m1 = __builtin_amdgcn_readfirstlane(wm1);
                unsigned r0 = rec0.x, r1 = rec0.y, slot0 = rec0.z;
                opaque_s(m0);
                opaque_s(m1);
                opaque_v(r0);
                opaque_v(r1);
                opaque_v(slot0);
                float *q = k->seis_t + ((size_t)s * k->d.nt + (it - 1)) * k->d.ngmax;
                const unsigned slot1 = slot0 + __popc(r0);
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const int b = c * R + r;
                        const unsigned bit = 1u << (b % 32);
                        const unsigned rm = b < 32 ? r0 : r1;
                        if (((b < 32 ? m0 : m1) & (int)bit) && (rm & bit))
                            q[(b < 32 ? slot0 : slot1) + __popc(rm & (bit - 1))] = p[c][r];
                    }
            }
            if (a.strips) {
                const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
                if (v_lane) {
                    float *q = sv + (v_slot * W + wave) * (C * R), *qw = q + 4 * W * C * R;
#pragma unroll
                    for (int c = 0; c < C; ++c)
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            q[c * R + r] = u[c][r];
                            qw[c * R + r] = w[c][r];
                        }
                }
                float *row = k->strips + ((size_t)s * k->s_rows + (it - 1) % k->s_rows) * k->d.S;
#pragma unroll
                for (int i = 0; i < NP; ++i)
                    if (sp_lds[i] >= 0) row[sp_slot[i]] = sp[sp_lds[i]];
                const int c1 = k->d.npml + 1 - x0, cn = k->d.npml + k->d.nx - x0;   // columns of jx = 1, nx
                if ((c1 >= -1 && c1 < C) || (cn >= 0 && cn <= C)) {
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        side_column(k, row, x0 + c, voff,
                                    c == c1 ? 0 : c == c1 + 1 ? 1 : c == cn ? 3 : c == cn - 1 ? 4 : -1, p[c]);
                        side_column(k, row, x0 + c, voff, c == c1 ? 2 : c == cn - 1 ? 5 : -1, u[c]);
                    }
                }
            }
            // ---- exchange, in: fresh halo columns ----
            if (edge && exch)
                recv_edges<FwdArgs, R, C>(has_l, has_r, wave, W, box, box + kMsg, tag, sh_place, dead, u);
            if (edge) __builtin_amdgcn_s_setprio(0);
            if constexpr (kLate) {
#pragma unroll
                for (int c = 0; c < C; ++c) store_hist(s, it, x0 + c, voff, hd[c]);
            }
            put_u();
            srcv = fresh_args<FwdArgs>()->d.dt * src_next;
            lds_barrier();
        }
        if (a.strips) copy_velocities(fresh_args<FwdArgs>(), s, it1 - 1);
        // state out: own columns
        if (a.out || a.end) {
            const ArgPtr<FwdArgs> k = fresh_args<FwdArgs>();
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            const int npml = k->d.npml, nx = k->d.nx, nz = k->d.nz, nzp = k->d.nzp, ld = k->d.ld;
            const int np = k->d.nxp * ld, ni = nx * nz;
            const int zr = k->c.z0 + (int)(voff >> 2), jz0 = zr - npml;
            const int os_ = window_os(k->c.W, C, j), oe_ = window_oe(k->c.W, C, j, k->c.P, k->d.nxp);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int x = x0 + c, jx = x - npml;
                if (x < os_ || x > oe_) continue;
                if (k->out) {
                    float *f = k->out + (size_t)s * 3 * np + (size_t)(x - 1) * ld;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (zr + r <= nzp) {
                            const unsigned o = zr + r - 1;
                            f[o] = p[c][r];
                            f[np + o] = u[c][r];
                            f[2 * np + o] = w[c][r];
                        }
                }
                if (k->end && jx >= 1 && jx <= nx) {
                    float *f = k->end + (size_t)s * 3 * ni + (size_t)(jx - 1) * nz;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (jz0 + r >= 1 && jz0 + r <= nz) {
                            const unsigned o = jz0 + r - 1;
                            f[o] = p[c][r];
                            f[ni + o] = u[c][r];
                            f[2 * ni + o] = w[c][r];
                        }
                }
            }
        }
        lds_barrier();               // the edges and the stage are rewritten by the next shot
    }
}

struct BwdArgs {
    Dims d;
    Cfg c;
    int s0, ns;                 // shots s0 .. s0 + ns - 1
    const float *co;            // coefficients as the forward's, adjoint regions (k_res_setup)
    int ncol;
    const float *fpx;
    const ShotGeom *geo;
    const float *src;           // [ns][nt]
    const void *strips;         // rows [ns][nt][S]
    int mode;                   // of the strips: 0 FP32, 1 FP16, 2 BF16
    const uint32_t *smax;
    const float *end;           // [ns][3][nx][nz] final forward state
    // adjoint sources: window w of shot s takes dt times values base[s][w] + n of
    // adj [ns][nt][ngmax]; n-th value's place in the injection stage itab [ns][P][2][64 W]
    const float *adj;
    const int *itab, *ibase;
    unsigned long long imask;   // lanes of the injection stage
    int layers;                 // receivers of one cell (1 or 2)
    int ring;                   // steps whose values are held (a power of two)
    int ninj, sides;            // most receivers, most side layers (1 or 2) of a window
    float *acc;                 // [ns][nxp][3][64 R] per-shot accumulators, zero at the start
    u64 *msg;                   // [G P][2 slots][2 sides][2 fields][3 R][64]
    Ctl *ctl;
    unsigned limit;             // as the forward's
};

// LDS of the backward: the waves' edge columns of both wavefields (p, then u: with R >= 5 in
// one place, with a barrier between the last read and the first write); two sets (a step's and
// the next one's) of the strip rows' lanes [4][W C][R], w of row nz-1 [W C], the injection
// stage [layers][NI + 1][W C][R] (the last one zeros); the values of `ring` steps as they
// come: [ring][6 W C strip values of the columns, ninj adjoint sources]; the side columns of
// `ring` steps [ring][sides][p, next p, u][64 R].
constexpr bool bwd_one_edge_set(int R) { return R >= 5; }
__host__ __device__ inline int bwd_edge_floats(int W, int R) { return W * (bwd_one_edge_set(R) ? 6 : 12) * R * 64; }
__host__ __device__ inline int bwd_set_floats(int W, int C, int R, int NI, int layers) {
    return 4 * W * C * R + ((W * C + 3) & ~3) + layers * (NI + 1) * W * C * R;
}
__host__ __device__ inline int bwd_step_floats(int W, int C, int R, int ninj, int sides) {
    return 6 * W * C + ninj + sides * 3 * 64 * R;
}

// Reverse steps nt .. 2 (solver.f90:230-253) of every shot: reconstruction (fdcore.f90:
// 202-289), adjoint step (:293-375) and imaging (solver.f90:237-239), both wavefields in
// registers (6 R C <= 150 floats at two waves per SIMD).  A step is: velocities of both
// fields from p (edges through LDS), strip values into the reconstructed u, w; then
// pressures, strip values into the reconstructed p, injection and mirror of the adjoint p,
// imaging.  Strip values and adjoint sources come from HBM, and loads complete in order: one
// value of the step that is fetched makes every later load of the wave wait for HBM.  So the
// values of ring - 1 steps are fetched at once, and handed out through LDS step by step.  The accumulators are read and written in memory every step (they stay in
// L2): the wavefields alone fill the registers.
// Per time step (481x141, 49 shots, in three rounds of 17; the step kernel 86 us): 33.9 us with
// values fetched one step ahead, 30.9 with the ring, 27.5 with the accumulators' loads and
// stores free of branches (a wait has to assume the fewest loads in flight that any path
// leaves, and so waited for the stores of the column before).  One shot of 201x81: 7.5 us by
// the step kernel, 6.4, 5.2, 5.1; 801x267, 81 shots: 432 by the step kernel, 224, 186, 180
// (R = 6: eight waves fit since the edges of p and u share their place).  Vector issue is 5.7 of
// the 9.2 us of a round of the 49 shots (counted: 103 instructions a padded cell).
template <int R, int C>
__global__ __launch_bounds__(512) void k_bwd_resident(BwdArgs a) {
    extern __shared__ float lds[];
    __shared__ unsigned sh_place[2];
    constexpr int kCol = 64 * R * 4;                     // bytes of a column of one array
    constexpr int NI6 = (6 * C + 63) / 64;               // strip values of the window's columns per thread
    const int W = a.c.W, P = a.c.P, T = W * 64;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) take_place(a.ctl, P, sh_place);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(sh_place[0]);
    const int grp = __builtin_amdgcn_readfirstlane(t / P), j = __builtin_amdgcn_readfirstlane(t % P);
    const int WC = W * C, NI = __popcll(a.imask);
    float *eP = lds;                                     // [W][2 fields][3][R][64]: first, second, last column of p
    // [W][2 fields][3][R][64]: first, last but one, last of u
    float *eU = bwd_one_edge_set(R) ? eP : eP + W * 6 * R * 64;
    const int set_floats = bwd_set_floats(W, C, R, NI, a.layers);
    const int ring = a.ring, nraw = 6 * WC + a.ninj;
    float *sets = lds + bwd_edge_floats(W, R);
    float *raw = sets + 2 * set_floats;
    float *side_ring = raw + ring * nraw;
    const int o_w = 4 * WC * R, o_inj = o_w + ((WC + 3) & ~3);
    const int xw = window_x(W, C, j), x0w = xw + wave * C;
    const bool has_l = j > 0, has_r = j + 1 < P;
    const bool edge = (has_l && wave <= (2 * kH - 1) / C) || (has_r && wave >= W - 1 - (2 * kH - 1) / C);
    const unsigned voff0 = lane * R * 4;
    const bool wave_pml = x0w <= a.d.npml || x0w + C - 1 >= a.d.npml + a.d.nx;
    const __amdgpu_buffer_rsrc_t co = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.co), 0, (int)((unsigned)(a.ncol + 1) * 5u * kCol), 0x00027000);
    unsigned tag = 0;
    bool dead = false;
    float fpz[R];
    buffer_rows<R>(co, voff0, 2 * kCol, fpz);
    // lanes of the mirror row fs-1 (their first row), of the strips' rows, of the injection
    const int lm = (a.d.fs - 1 - a.c.z0) / R;
    const int lb = (a.d.npml + a.d.nz - 1 - a.c.z0) / R;           // row nz - 1
    const bool mir_lane = lane == lm, mir_w = a.d.free_surface == 1 && lane == lm;
    const int b_slot = lane <= lm + 1 ? max(lane - lm, 0) : min(max(lane - lb, 0) + 2, 3);
    const int i_slot = (a.imask >> lane) & 1 ? __popcll(a.imask & ((1ull << lane) - 1)) : NI;
    // rows of this lane: bit r: a strip row (jz 1..3, nz-1, nz); row nz - 1; bit: any interior row
    unsigned brow = 0, wrow = 0;
    bool inner = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int jz = a.c.z0 + lane * R + r - a.d.npml;
        if ((jz >= 1 && jz <= 3) || jz == a.d.nz - 1 || jz == a.d.nz) brow |= 1u << r;
        if (jz == a.d.nz - 1) wrow |= 1u << r;
        inner = inner || (jz >= 1 && jz <= a.d.nz);
    }
    const unsigned acc_off = inner ? voff0 : 0x80000000u;          // past the buffer: loads 0, stores nothing

    // ---- values of a step: strip values of the window's columns (n-th: column n / 6, value
    // n % 6: p of jz = 1, 2, 3, nz, nz-1, w of nz-1), the thread's own at n = tid + i T, to
    // place col_dst of a set; adjoint sources; side columns ----
    int col_dst[NI6];
    {
        const int nx = a.d.nx, nz = a.d.nz, npml = a.d.npml;
#pragma unroll
        for (int i = 0; i < NI6; ++i) {
            const int n = threadIdx.x + i * T, col = n / 6, q = n % 6, jx = xw + col - npml;
            const int row = (q < 3 ? q + 1 : q == 3 ? nz : nz - 1) + npml - a.c.z0, L = row / R;
            col_dst[i] = col >= WC || jx < 1 || jx > nx ? -1
                         : q == 5                       ? o_w + col
                                                        : ((L <= lm + 1 ? L - lm : 2 + L - lb) * WC + col) * R + row % R;
        }
    }
    const bool side_l = xw <= a.d.npml + 2 && xw + WC > a.d.npml + 1;
    const bool side_r = xw <= a.d.npml + a.d.nx && xw + WC > a.d.npml + a.d.nx - 1;
    constexpr int kSide = 64 * R;
    const int side_floats = a.sides * 3 * kSide, o_right = side_l ? 3 * kSide : 0;
    const int c1 = a.d.npml + 1 - x0w, cn = a.d.npml + a.d.nx - x0w;      // this wave's columns of jx = 1, nx
    const bool wave_side = (c1 < C && c1 >= -1) || (cn >= 0 && cn <= C);
    // values of steps t, t-1, .. (ring - 1 of them, down to step 2) into the ring
    auto fetch_steps = [&](int s, int t, int i0, int i1, int ib) {
        constexpr int U = 4;                             // steps in flight
        const ArgPtr<BwdArgs> k = fresh_args<BwdArgs>();
        const int nx = k->d.nx, nz = k->d.nz, mode = k->mode, WC_ = k->c.W * C, T_ = k->c.W * 64;
        const size_t S = k->d.S, row0 = (size_t)s * k->d.nt + (t - 2), ngmax = k->d.ngmax;
        const int cnt = min(ring - 1, t - 1);
        unsigned tid = threadIdx.x;
        opaque_v(tid);
        auto get = [&](size_t i, float scale) -> float {
            if (mode == 0) return ((const float *)k->strips)[i];
            const uint16_t x = ((const uint16_t *)k->strips)[i];
            return (mode == 1 ? strip_decode<1>(x) : strip_decode<2>(x)) * scale;
        };
        // lane l: the scale of the l-th row (16-bit strips)
        const float scales = mode ? strip_scale(k->smax[row0 - min(lane, cnt - 1)]) : 1.0f;
        auto scale_of = [&](int n) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(scales), n)); };
        const float *adj = k->adj + (row0 + 1) * ngmax + ib + tid;
        for (int b = 0; b < cnt; b += U) {
            float v[U][NI6], g0[U], g1[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (b + u >= cnt) break;
                const size_t row = row0 - (b + u);
                const float scale = scale_of(b + u);
#pragma unroll
                for (int i = 0; i < NI6; ++i) {
                    const int n = tid + i * T_, col = n / 6, q = n % 6, jx = window_x(k->c.W, C, j) + col - k->d.npml;
                    v[u][i] = 0.0f;
                    if (col < WC_ && jx >= 1 && jx <= nx)
                        v[u][i] = get(row * S + (q < 3 ? 3 * nx + 6 * nz + 6 * (jx - 1) + q : 3 * (jx - 1) + q - 3), scale);
                }
                g0[u] = i0 >= 0 ? adj[0] : 0.0f;
                g1[u] = i1 >= 0 ? adj[T_] : 0.0f;
                adj -= ngmax;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (b + u >= cnt) break;
                float *q = raw + ((t - b - u) & (ring - 1)) * nraw + tid;
#pragma unroll
                for (int i = 0; i < NI6; ++i)
                    if ((int)tid + i * T_ < 6 * WC_) q[i * T_] = v[u][i];
                if (i0 >= 0) q[6 * WC_] = k->d.dt * g0[u];
                if (i1 >= 0) q[6 * WC_ + T_] = k->d.dt * g1[u];
            }
        }
        if (side_l || side_r) {
            const int n1 = side_l && side_r ? 2 * kSide : kSide;
            for (int n = tid; n < n1; n += T_) {
                const int right = side_l ? n / kSide : 1, row_ = n % kSide, jz = k->c.z0 + row_ - k->d.npml;
                if (jz < 1 || jz > nz) continue;
                const size_t o = 3 * nx + 6 * (jz - 1) + 3 * right;
                float *to = side_ring + (right ? o_right : 0) + row_;
                for (int b = 0; b < cnt; b += U) {
                    float v[U][3];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        if (b + u >= cnt) break;
                        const size_t row = row0 - (b + u);
                        const float scale = scale_of(b + u);
#pragma unroll
                        for (int q = 0; q < 3; ++q) v[u][q] = get(row * S + o + q, scale);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        if (b + u >= cnt) break;
                        float *f = to + ((t - b - u) & (ring - 1)) * side_floats;
#pragma unroll
                        for (int q = 0; q < 3; ++q) f[q * kSide] = v[u][q];
                    }
                }
            }
        }
    };
    // step t's own values from the ring into its set
    auto hand_out = [&](int t, int i0, int i1) {
        float *f = sets + (t & 1) * set_floats;
        const float *q = raw + (t & (ring - 1)) * nraw + threadIdx.x;
#pragma unroll
        for (int i = 0; i < NI6; ++i)
            if (col_dst[i] >= 0) f[col_dst[i]] = q[i * T];
        if (i0 >= 0) f[o_inj + i0] = q[6 * WC];
        if (i1 >= 0) f[o_inj + i1] = q[6 * WC + T];
    };

    for (int s = a.s0 + grp; s < a.s0 + a.ns; s += a.c.G) {
        const int isx = a.geo[s].isx_i + a.d.npml, isz = a.geo[s].isz_i + a.d.npml;   // padded cell
        const bool src_in = a.geo[s].isx_i > 2 && a.geo[s].isx_i < a.d.nx - 1 && a.geo[s].isz_i > 3 &&
                            a.geo[s].isz_i < a.d.nz - 1;
        const float *src = a.src + (size_t)s * a.d.nt;
        const int i0 = a.itab[((size_t)s * P + j) * 2 * T + threadIdx.x];
        const int i1 = a.itab[((size_t)s * P + j) * 2 * T + T + threadIdx.x];
        const int ib = a.ibase[s * P + j];
        for (int i = threadIdx.x; i < 2 * set_floats + ring * (nraw + side_floats); i += T) sets[i] = 0.0f;
        float pr[C][R], ur[C][R], wr[C][R], pa[C][R], ua[C][R], wa[C][R];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int r = 0; r < R; ++r) pr[c][r] = ur[c][r] = wr[c][r] = pa[c][r] = ua[c][r] = wa[c][r] = 0.0f;
        {
            const ArgPtr<BwdArgs> k = fresh_args<BwdArgs>();
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            const int npml = k->d.npml, nx = k->d.nx, nz = k->d.nz, ni = nx * nz;
            const int jz0 = k->c.z0 + (int)(voff >> 2) - npml;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int jx = x0 + c - npml;
                if (jx < 1 || jx > nx) continue;
                const float *f = k->end + (size_t)s * 3 * ni + (size_t)(jx - 1) * nz;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (jz0 + r < 1 || jz0 + r > nz) continue;
                    const unsigned o = jz0 + r - 1;
                    pr[c][r] = f[o];
                    ur[c][r] = f[ni + o];
                    wr[c][r] = f[2 * ni + o];
                }
            }
        }
        __syncthreads();
        int left = a.d.nt;                               // first step whose values are not fetched
        fetch_steps(s, left, i0, i1, ib);
        left -= ring - 1;
        hand_out(a.d.nt, i0, i1);
        // p of the edge columns for the next step
        auto put_p = [&]() {
            float *e = eP + (size_t)wave * 6 * R * 64 + lane;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                e[r * 64] = pr[0][r];
                e[(R + r) * 64] = pr[1][r];
                e[(2 * R + r) * 64] = pr[C - 1][r];
                e[(3 * R + r) * 64] = pa[0][r];
                e[(4 * R + r) * 64] = pa[1][r];
                e[(5 * R + r) * 64] = pa[C - 1][r];
            }
        };
        // edge column `q` (0, 1, 2; + 3 for the adjoint) of a neighbouring wave, zero past the window
        auto edge_rows = [&](const float *e, int w, int q, float (&v)[R]) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                v[r] = w >= 0 && w < W ? e[((w * 6 + q) * R + r) * 64 + lane] : 0.0f;
        };
        put_p();
        lds_barrier();
        for (int it = a.d.nt; it >= 2; --it) {
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            const float *set = sets + (it & 1) * set_floats;
            if (it - 1 == left && it > 2) {
                fetch_steps(s, left, i0, i1, ib);
                left -= ring - 1;
            }
            const float *side = side_ring + (it & (ring - 1)) * side_floats + voff / 4;
            float ssub;                                  // the reference's s(it+1), 0 past the end
            {
                const ArgPtr<BwdArgs> k = fresh_args<BwdArgs>();
                ssub = it + 1 <= k->d.nt ? k->d.dt * src[it] : 0.0f;
            }
            // ---- velocities: reconstruction (:221-247), adjoint (:310-326) ----
            {
                float kp[2][R], kv[2][R], fu[2][R], fw[2][R];
                auto fetch = [&](int c) {
                    const int f = wave_pml ? (x0 + c) * (5 * kCol) : 0;
                    buffer_rows<R>(co, voff, (x0 + c) * (5 * kCol), kp[c & 1]);
                    buffer_rows<R>(co, voff, (x0 + c) * (5 * kCol) + kCol, kv[c & 1]);
                    buffer_rows<R>(co, voff, f + 3 * kCol, fu[c & 1]);
                    buffer_rows<R>(co, voff, f + 4 * kCol, fw[c & 1]);
                };
                fetch(0);
                float rl[R], al[R], r1[R], a1[R], r2[R], a2[R];
                edge_rows(eP, wave - 1, 2, rl);
                edge_rows(eP, wave - 1, 5, al);
                edge_rows(eP, wave + 1, 0, r1);
                edge_rows(eP, wave + 1, 3, a1);
                edge_rows(eP, wave + 1, 1, r2);
                edge_rows(eP, wave + 1, 4, a2);
                if constexpr (bwd_one_edge_set(R)) lds_barrier();
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if (c + 1 < C) fetch(c + 1);
                    {
                        const float pd = dn1(pr[c][R - 1]), pu0 = up1(pr[c][0]), pu1 = up1(pr[c][1]);
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const float xm = c >= 1 ? pr[c - (c >= 1)][r] : rl[r];
                            const float xp = c + 1 < C ? pr[c + (c + 1 < C)][r] : r1[r];
                            const float xq = c + 2 < C ? pr[c + (c + 2 < C ? 2 : 0)][r] : c + 2 == C ? r1[r] : r2[r];
                            const float zm = r >= 1 ? pr[c][r - (r >= 1)] : pd;
                            const float zp = r + 1 < R ? pr[c][r + (r + 1 < R)] : pu0;
                            const float zq = r + 2 < R ? pr[c][r + (r + 2 < R ? 2 : 0)] : r + 2 == R ? pu0 : pu1;
                            ur[c][r] = v_undo(ur[c][r], kp[c & 1][r], pr[c][r], xp, xq, xm);
                            wr[c][r] = v_undo(wr[c][r], kp[c & 1][r], pr[c][r], zp, zq, zm);
                        }
                    }
                    {
                        const float pd = dn1(pa[c][R - 1]), pu0 = up1(pa[c][0]), pu1 = up1(pa[c][1]);
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const float xm = c >= 1 ? pa[c - (c >= 1)][r] : al[r];
                            const float xp = c + 1 < C ? pa[c + (c + 1 < C)][r] : a1[r];
                            const float xq = c + 2 < C ? pa[c + (c + 2 < C ? 2 : 0)][r] : c + 2 == C ? a1[r] : a2[r];
                            const float zm = r >= 1 ? pa[c][r - (r >= 1)] : pd;
                            const float zp = r + 1 < R ? pa[c][r + (r + 1 < R)] : pu0;
                            const float zq = r + 2 < R ? pa[c][r + (r + 2 < R ? 2 : 0)] : r + 2 == R ? pu0 : pu1;
                            ua[c][r] = v_update_f(ua[c][r], kv[c & 1][r], fu[c & 1][r], pa[c][r], xp, xq, xm);
                            wa[c][r] = v_update_f(wa[c][r], kv[c & 1][r], fw[c & 1][r], pa[c][r], zp, zq, zm);
                        }
                    }
                    if (mir_w) wa[c][0] = wa[c][1];
                    // strip value of the reconstructed w, row nz - 1
                    const float ws = set[o_w + wave * C + c];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        if (wrow & (1u << r)) wr[c][r] = ws;
                        pin(ur[c][r]);
                        pin(wr[c][r]);
                        pin(ua[c][r]);
                        pin(wa[c][r]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // strip values of the reconstructed u, columns jx = 1 and nx - 1
            if (wave_side) {
#pragma unroll
                for (int c = 0; c < C; ++c)
                    if (c == c1 || c == cn - 1) {
                        const float *q = side + (c == c1 ? 0 : o_right) + 2 * kSide;
#pragma unroll
                        for (int r = 0; r < R; ++r) ur[c][r] = q[r];
                    }
            }
            {
                float *e = eU + (size_t)wave * 6 * R * 64 + lane;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    e[r * 64] = ur[0][r];
                    e[(R + r) * 64] = ur[C - 2][r];
                    e[(2 * R + r) * 64] = ur[C - 1][r];
                    e[(3 * R + r) * 64] = ua[0][r];
                    e[(4 * R + r) * 64] = ua[C - 2][r];
                    e[(5 * R + r) * 64] = ua[C - 1][r];
                }
            }
            // the reconstruction's source subtraction
            if (src_in && (unsigned)(isx - x0) < (unsigned)C) {
                const int zr = fresh_args<BwdArgs>()->c.z0 + (int)(voff >> 2);
#pragma unroll
                for (int c = 0; c < C; ++c)
                    if (x0 + c == isx) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            if (zr + r == isz) pr[c][r] = pr[c][r] - ssub;
                    }
            }
            lds_barrier();
            // ---- pressures: reconstruction (:250-287), adjoint (:336-373), imaging ----
            if (edge) __builtin_amdgcn_s_setprio(3);
            {
                const ArgPtr<BwdArgs> k = fresh_args<BwdArgs>();
                const ArgPtr<float> fpx = (ArgPtr<float>)k->fpx + x0;
                const int os = window_os(k->c.W, C, j), oe = window_oe(k->c.W, C, j, k->c.P, k->d.nxp);
                const int ca = max(c1, os - x0), cb = min(cn, oe - x0);             // columns imaged here
                const __amdgpu_buffer_rsrc_t ab = __builtin_amdgcn_make_buffer_rsrc(
                    k->acc + (size_t)s * k->d.nxp * (3 * 64 * R), 0, (int)((unsigned)k->d.nxp * 3u * kCol), 0x00027000);
                const unsigned ao = voff + (acc_off - voff0);
                float kp[2][R], kv[2][R], g0[2][R], g1[2][R], g2[2][R];
                auto fetch = [&](int c) {
                    buffer_rows<R>(co, voff, (x0 + c) * (5 * kCol), kp[c & 1]);
                    buffer_rows<R>(co, voff, (x0 + c) * (5 * kCol) + kCol, kv[c & 1]);
                    // no branch (the loads and stores in flight stay countable): past the buffer
                    // where nothing is imaged
                    const bool im = c >= ca && c <= cb;
                    const int o = im ? (x0 + c - 1) * (3 * kCol) : 0;
                    const unsigned aoc = ao | (im ? 0u : 0x80000000u);
                    buffer_rows<R>(ab, aoc, o, g0[c & 1]);
                    buffer_rows<R>(ab, aoc, o + kCol, g1[c & 1]);
                    buffer_rows<R>(ab, aoc, o + 2 * kCol, g2[c & 1]);
                };
                fetch(0);
                float r2[R], a2[R], r1[R], a1[R], rr[R], ar[R];
                edge_rows(eU, wave - 1, 1, r2);
                edge_rows(eU, wave - 1, 4, a2);
                edge_rows(eU, wave - 1, 2, r1);
                edge_rows(eU, wave - 1, 5, a1);
                edge_rows(eU, wave + 1, 0, rr);
                edge_rows(eU, wave + 1, 3, ar);
                if constexpr (bwd_one_edge_set(R)) lds_barrier();
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if (c + 1 < C) fetch(c + 1);
                    const float fx = fpx[c];
                    {
                        const float wd1 = dn1(wr[c][R - 1]), wd2 = dn1(wr[c][R - 2]), wu = up1(wr[c][0]);
                        const float *q = set + (b_slot * WC + wave * C + c) * R;
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const float um1 = c >= 1 ? ur[c - (c >= 1)][r] : r1[r];
                            const float um2 = c >= 2 ? ur[c - (c >= 2 ? 2 : 0)][r] : c == 1 ? r1[r] : r2[r];
                            const float up = c + 1 < C ? ur[c + (c + 1 < C)][r] : rr[r];
                            const float wm1 = r >= 1 ? wr[c][r - (r >= 1)] : wd1;
                            const float wm2 = r >= 2 ? wr[c][r - (r >= 2 ? 2 : 0)] : r == 1 ? wd1 : wd2;
                            const float wp1 = r + 1 < R ? wr[c][r + (r + 1 < R)] : wu;
                            const float v = p_undo(pr[c][r], kv[c & 1][r], ur[c][r], um1, up, um2, wr[c][r], wm1, wp1,
                                                   wm2);
                            pr[c][r] = brow & (1u << r) ? q[r] : v;
                        }
                    }
                    if (wave_side && (c == c1 || c == c1 + 1 || c == cn - 1 || c == cn)) {
                        const float *q = side + (c == c1 || c == c1 + 1 ? 0 : o_right) + (c == c1 || (c != c1 + 1 && c == cn) ? 0 : kSide);
#pragma unroll
                        for (int r = 0; r < R; ++r) pr[c][r] = q[r];
                    }
                    float old[R];
                    {
                        const float wd1 = dn1(wa[c][R - 1]), wd2 = dn1(wa[c][R - 2]), wu = up1(wa[c][0]);
                        const float *q = set + o_inj + (i_slot * WC + wave * C + c) * R;
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            const float um1 = c >= 1 ? ua[c - (c >= 1)][r] : a1[r];
                            const float um2 = c >= 2 ? ua[c - (c >= 2 ? 2 : 0)][r] : c == 1 ? a1[r] : a2[r];
                            const float up = c + 1 < C ? ua[c + (c + 1 < C)][r] : ar[r];
                            const float wm1 = r >= 1 ? wa[c][r - (r >= 1)] : wd1;
                            const float wm2 = r >= 2 ? wa[c][r - (r >= 2 ? 2 : 0)] : r == 1 ? wd1 : wd2;
                            const float wp1 = r + 1 < R ? wa[c][r + (r + 1 < R)] : wu;
                            old[r] = pa[c][r];
                            pa[c][r] = p_update_f(pa[c][r], kp[c & 1][r], fminf(fx, fpz[r]), ua[c][r], um1, up, um2,
                                                  wa[c][r], wm1, wp1, wm2);
                            pa[c][r] = pa[c][r] + q[r];
                        }
                        if (k->layers > 1) {
                            const float *q2 = q + (NI + 1) * WC * R;
#pragma unroll
                            for (int r = 0; r < R; ++r) pa[c][r] = pa[c][r] + q2[r];
                        }
                        const float pm = R > 2 ? pa[c][R > 2 ? 2 : 0] : up1(pa[c][0]);
                        if (mir_lane) pa[c][0] = -pm;
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        pin(pr[c][r]);
                        pin(pa[c][r]);
                    }
                    {
                        const bool im = c >= ca && c <= cb;
                        const int o = im ? (x0 + c - 1) * (3 * kCol) : 0;
                        const unsigned aoc = ao | (im ? 0u : 0x80000000u);
#pragma unroll
                        for (int r = 0; r < R; ++r) {
                            g0[c & 1][r] = g0[c & 1][r] + pr[c][r] * (old[r] - pa[c][r]);
                            g1[c & 1][r] = g1[c & 1][r] + pr[c][r] * pr[c][r];
                            g2[c & 1][r] = g2[c & 1][r] + pa[c][r] * pa[c][r];
                        }
                        buffer_store_rows<R>(ab, aoc, o, g0[c & 1]);
                        buffer_store_rows<R>(ab, aoc, o + kCol, g1[c & 1]);
                        buffer_store_rows<R>(ab, aoc, o + 2 * kCol, g2[c & 1]);
                        after_stores<R>(g0[c & 1], g1[c & 1], g2[c & 1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // ---- exchange of p, the next step's values ----
            const bool exch = it > 2;
            if (exch) ++tag;
            constexpr int kMsg = 2 * kH * R * 64;
            u64 *box = nullptr;
            if (edge && exch) {
                const ArgPtr<BwdArgs> k = fresh_args<BwdArgs>();
                box = k->msg + ((size_t)(grp * k->c.P + j) * 2 + (tag & 1)) * (2 * kMsg) + voff / (4 * R);
                send_edges<R, C>(has_l, has_r, wave, W, box - 3 * kMsg, box + 4 * kMsg, tag, pr);
                send_edges<R, C>(has_l, has_r, wave, W, box - 3 * kMsg + kMsg / 2, box + 4 * kMsg + kMsg / 2, tag, pa);
            }
            if (exch) hand_out(it - 1, i0, i1);
            if (edge && exch) {
                recv_edges<BwdArgs, R, C>(has_l, has_r, wave, W, box, box + kMsg, tag, sh_place, dead, pr);
                recv_edges<BwdArgs, R, C>(has_l, has_r, wave, W, box + kMsg / 2, box + kMsg + kMsg / 2, tag, sh_place,
                                          dead, pa);
            }
            if (edge) __builtin_amdgcn_s_setprio(0);
            put_p();
            lds_barrier();
        }
    }
}

// Cross-shot FP64 sum of the resident backward's accumulators and g = -2 g / c (as
// k_reduce_acc); NaN if a wait of the job, or of the forward whose strips it used, ran out.
__global__ void k_res_reduce(Dims d, int ns, int R, int z0, const float *__restrict__ vp, const float *__restrict__ acc,
                             double *__restrict__ grad, double *__restrict__ fw, double *__restrict__ bk,
                             const Ctl *ctl) {
    const int jz = blockIdx.x * blockDim.x + threadIdx.x + 1, jx = blockIdx.y * blockDim.y + threadIdx.y + 1;
    if (jz > d.nz || jx > d.nx) return;
    const size_t n = (size_t)64 * R, per = (size_t)d.nxp * 3 * n;
    const float *p = acc + (size_t)(jx + d.npml - 1) * 3 * n + (jz + d.npml - z0);
    double g = 0.0, f = 0.0, b = 0.0;
    for (int s = 0; s < ns; ++s, p += per) {
        g += (double)p[0];
        f += (double)p[n];
        b += (double)p[2 * n];
    }
    const size_t k = iidx(d, jz, jx);
    if (ctl->err | ctl->bad[kStrips]) g = f = b = __builtin_nan("");
    grad[k] = -2.0 * g / (double)vp[k];
    fw[k] = f;
    bk[k] = b;
}

// Adjoint sources into slot order: out[s][t][n] = in[s][map[s][n]][t] (map -1: nothing).
__global__ void k_res_adjsrc(int nt, int ngmax, const int *__restrict__ map, const float *__restrict__ in,
                             float *__restrict__ out) {
    __shared__ float tile[32][33];
    const int s = blockIdx.z, n0 = blockIdx.x * 32, t0 = blockIdx.y * 32;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int n = n0 + k, t = t0 + threadIdx.x;
        const int m = n < ngmax ? map[(size_t)s * ngmax + n] : -1;
        if (m >= 0 && t < nt) tile[k][threadIdx.x] = in[((size_t)s * ngmax + m) * nt + t];
    }
    __syncthreads();
    const int n = n0 + threadIdx.x;
    const int m = n < ngmax ? map[(size_t)s * ngmax + n] : -1;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int t = t0 + k;
        if (m >= 0 && t < nt) out[((size_t)s * nt + t) * ngmax + n] = tile[threadIdx.x][k];
    }
}


struct ExArgs {
    Dims d;
    Cfg c;
    int ns;
    int it0, it1;               // reverse steps it1 .. it0
    const float *co;            // the forward's coefficients (k_res_setup)
    int ncol;
    const float *fpx;
    const float *g;             // [ns][nt][ngmax] dJ/dseis
    const int2 *itab;           // [ns][P][2][64 W] {place in the injection stage, receiver}, -1 none
    unsigned long long imask;   // lanes of the injection stage
    int layers;                 // most receivers of one cell (1 or 2)
    DSave hist;                 // divergence history
    const float *in;            // null (zero state) or [ns][3][nxp][ld]: adjoint fields after step it1 + 1
    float *out;                 // null or [ns][3][nxp][ld]
    float *gk;                  // [ns][nxp][ld] K-gradient so far, zero outside the p region
    int add;                    // 0: it is zero
    u64 *msg;                   // as the forward's
    Ctl *ctl;
    unsigned limit;
};

// LDS of the exact reverse loop: the waves' edge columns of q and r, two injection stages.
__host__ __device__ inline int ex_set_floats(int W, int C, int R, int NI, int layers) { return layers * NI * W * C * R; }

// Reverse steps it1 .. it0 of the exact adjoint (the transpose of the forward step, written
// out in fd_exact.hip) of every shot, the three adjoint fields, the K-gradient, K and B in
// registers.  qu = B lu takes the place of the forward's u and r = K lp that of its p: lp
// needs qu at x-2..x+1 and lu needs r at x-1..x+2, so fresh lu in the halo after every step
// keeps the rest that is needed right, receivers in the halo included.
// Bound by vector issue, 34 operations per cell and step and about as many again for shifts,
// the divergence history (one 4-byte load per cell and step, in flight through the first
// part) and the exchange.  Forward and reverse of 161x61x1500, 8 shots, whole history: 31.2 ms
// by the step kernels (a launch each per step), 8.5 ms here; of 301x101, 21 shots, with
// checkpoints (an additional forward): 81.8 and 18.5 ms.
template <int R, int C>
__global__ __launch_bounds__(512) void k_ex_resident(ExArgs a) {
    extern __shared__ float lds[];
    __shared__ unsigned sh_place[2];
    constexpr int kCol = 64 * R * 4;
    const int W = a.c.W, P = a.c.P, T = W * 64;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) take_place(a.ctl, P, sh_place);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(sh_place[0]);
    const int grp = __builtin_amdgcn_readfirstlane(t / P), j = __builtin_amdgcn_readfirstlane(t % P);
    const int NI = __popcll(a.imask);
    float *eQ = lds;                                     // [W][3][R][64]: first, last but one, last column of qu
    float *eR = eQ + W * 3 * R * 64;                     // [W][3][R][64]: first, second, last column of r
    float *sets = eR + W * 3 * R * 64;
    const int set_floats = ex_set_floats(W, C, R, NI, a.layers), layer_floats = NI * W * C * R;
    const int x0w = window_x(W, C, j) + wave * C;
    const bool has_l = j > 0, has_r = j + 1 < P;
    const bool edge = (has_l && wave <= (2 * kH - 1) / C) || (has_r && wave >= W - 1 - (2 * kH - 1) / C);
    const unsigned voff0 = lane * R * 4;
    const bool mirror = a.d.free_surface == 1 && lane == 0;
    const bool mirror1 = a.d.free_surface == 1 && lane == 1;
    const bool wave_pml = x0w <= a.d.npml || x0w + C - 1 >= a.d.npml + a.d.nx;
    const __amdgpu_buffer_rsrc_t co = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.co), 0, (int)((unsigned)(a.ncol + 1) * 5u * kCol), 0x00027000);
    const bool i_lane = (a.imask >> lane) & 1;
    const int i_off = (__popcll(a.imask & ((1ull << lane) - 1)) * W + wave) * (C * R);
    unsigned tag = 0;
    bool dead = false;
    float K[C][R], B[C][R], fpz[R];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        buffer_rows<R>(co, voff0, (x0w + c) * (5 * kCol), K[c]);
        buffer_rows<R>(co, voff0, (x0w + c) * (5 * kCol) + kCol, B[c]);
    }
    buffer_rows<R>(co, voff0, 2 * kCol, fpz);

    for (int s = grp; s < a.ns; s += a.c.G) {
        float lp[C][R], lu[C][R], lw[C][R], gk[C][R];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int r = 0; r < R; ++r) lp[c][r] = lu[c][r] = lw[c][r] = gk[c][r] = 0.0f;
        if (a.in || a.add) {
            const ArgPtr<ExArgs> k = fresh_args<ExArgs>();
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            const int zr = k->c.z0 + (int)(voff >> 2), ld = k->d.ld, np = k->d.nxp * ld;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                if (x0 + c > k->d.nxp) continue;
                const float *f = k->in + (size_t)s * 3 * np + (size_t)(x0 + c - 1) * ld;
                const float *g = k->gk + (size_t)s * np + (size_t)(x0 + c - 1) * ld;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (zr + r > k->d.nzp) continue;
                    const unsigned o = zr + r - 1;
                    if (k->in) {
                        lp[c][r] = f[o];
                        lu[c][r] = f[np + o];
                        lw[c][r] = f[2 * np + o];
                    }
                    if (k->add) gk[c][r] = g[o];
                }
            }
        }
        const int2 *tab = a.itab + ((size_t)s * P + j) * 2 * T + threadIdx.x;
        const int2 i0 = tab[0], i1 = tab[T];
        for (int n = threadIdx.x; n < 2 * set_floats; n += T) sets[n] = 0.0f;
        // qu of the edge columns for the next step
        auto put_q = [&]() {
            float *e = eQ + (size_t)wave * 3 * R * 64 + lane;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                e[r * 64] = B[0][r] * lu[0][r];
                e[(R + r) * 64] = B[C - 2][r] * lu[C - 2][r];
                e[(2 * R + r) * 64] = B[C - 1][r] * lu[C - 1][r];
            }
        };
        __syncthreads();
        const int ngmax = a.d.ngmax;
        const float *grow = a.g + ((size_t)s * a.d.nt + (a.it1 - 1)) * ngmax;
        {
            float *f = sets + (a.it1 & 1) * set_floats;
            if (i0.x >= 0) f[i0.x] = grow[i0.y];
            if (i1.x >= 0) f[i1.x] = grow[i1.y];
        }
        put_q();
        __syncthreads();
        const int it0 = a.it0;
        for (int it = a.it1; it >= it0; --it) {
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            // D(it) of the window's columns (past the grid: the last column's, for cells that
            // are never stored) and the next step's injection
            float D[C][R];
            {
                const ArgPtr<ExArgs> k = fresh_args<ExArgs>();
                const int ld = k->d.ld, nxp = k->d.nxp, np = nxp * ld;
                const __amdgpu_buffer_rsrc_t h = __builtin_amdgcn_make_buffer_rsrc(
                    k->hist.p + ((size_t)s * k->hist.slots + (it - 1 - k->hist.base)) * np, 0, np * 4, 0x00027000);
                const unsigned zo = voff + (k->c.z0 - 1) * 4;
#pragma unroll
                for (int c = 0; c < C; ++c) buffer_rows<R>(h, zo, (min(x0 + c, nxp) - 1) * ld * 4, D[c]);
            }
            grow -= ngmax;
            float gn0 = 0.0f, gn1 = 0.0f;
            if (it > it0) {
                if (i0.x >= 0) gn0 = grow[i0.y];
                if (i1.x >= 0) gn1 = grow[i1.y];
            }
            // ---- lp += g at the receivers, in receiver order ----
            if (i_lane) {
                const float *q = sets + (it & 1) * set_floats + i_off;
                for (int l = a.layers; l > 0; --l, q += layer_floats) {
#pragma unroll
                    for (int c = 0; c < C; ++c)
#pragma unroll
                        for (int r = 0; r < R; ++r) lp[c][r] = lp[c][r] + q[c * R + r];
                }
            }
            // ---- lp -= Gx^T qu + Gz^T qw; gK -= lp D; qu of the columns x0-2, x0-1, x0+C ----
            {
                float ql2[R], ql1[R], qr1[R], q[C][R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float *e = eQ + lane;
                    ql2[r] = wave > 0 ? e[(((wave - 1) * 3 + 1) * R + r) * 64] : 0.0f;
                    ql1[r] = wave > 0 ? e[(((wave - 1) * 3 + 2) * R + r) * 64] : 0.0f;
                    qr1[r] = wave + 1 < W ? e[((wave + 1) * 3 * R + r) * 64] : 0.0f;
                    q[0][r] = B[0][r] * lu[0][r];
                }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if (c + 1 < C) {
#pragma unroll
                        for (int r = 0; r < R; ++r) q[c + (c + 1 < C)][r] = B[c + (c + 1 < C)][r] * lu[c + (c + 1 < C)][r];
                    }
                    // w mirror transposed: rows fs-1, fs are lane 0's first two
                    const float wf = lw[c][1] + lw[c][0];
                    lw[c][1] = mirror ? wf : lw[c][1];
                    lw[c][0] = mirror ? 0.0f : lw[c][0];
                    float qw[R];
#pragma unroll
                    for (int r = 0; r < R; ++r) qw[r] = B[c][r] * lw[c][r];
                    const float d1 = dn1(qw[R - 1]), d2 = dn1(qw[R - 2]), un = up1(qw[0]);
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float xm1 = c >= 1 ? q[c - (c >= 1)][r] : ql1[r];
                        const float xm2 = c >= 2 ? q[c - (c >= 2 ? 2 : 0)][r] : c == 1 ? ql1[r] : ql2[r];
                        const float xp1 = c + 1 < C ? q[c + (c + 1 < C)][r] : qr1[r];
                        const float zm1 = r >= 1 ? qw[r - (r >= 1)] : d1;
                        const float zm2 = r >= 2 ? qw[r - (r >= 2 ? 2 : 0)] : r == 1 ? d1 : d2;
                        const float zp1 = r + 1 < R ? qw[r + (r + 1 < R)] : un;
                        const float gx = kC1 * (xm1 - q[c][r]) + kC2 * (xm2 - xp1);
                        const float gz = kC1 * (zm1 - qw[r]) + kC2 * (zm2 - zp1);
                        lp[c][r] = lp[c][r] - gx - gz;
                    }
                    // p mirror transposed: row fs+1 (lane 1's first when R = 2) -= row fs-1
                    if constexpr (R > 2) {
                        const float pf = lp[c][R > 2 ? 2 : 0] - lp[c][0];
                        lp[c][R > 2 ? 2 : 0] = mirror ? pf : lp[c][R > 2 ? 2 : 0];
                    } else {
                        const float pf = lp[c][0] - dn1(lp[c][0]);
                        lp[c][0] = mirror1 ? pf : lp[c][0];
                    }
                    lp[c][0] = mirror ? 0.0f : lp[c][0];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        gk[c][r] = gk[c][r] - lp[c][r] * D[c][r];
                        pin(lp[c][r]);
                        pin(lw[c][r]);
                        pin(gk[c][r]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // ---- r = K lp; lu -= Dx^T r, lw -= Dz^T r; lp *= fp; r of x0-1, x0+C, x0+C+1 ----
            float cfu[2][R], cfw[2][R];
            auto fetch_v = [&](int c) {
                const int f = wave_pml ? (x0 + c) * (5 * kCol) : 0;
                buffer_rows<R>(co, voff, f + 3 * kCol, cfu[c % 2]);
                buffer_rows<R>(co, voff, f + 4 * kCol, cfw[c % 2]);
            };
            fetch_v(0);
            float rc[C][R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                rc[0][r] = K[0][r] * lp[0][r];
                rc[1][r] = K[1][r] * lp[1][r];
            }
            {
                float *e = eR + (size_t)wave * 3 * R * 64 + lane;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    e[r * 64] = rc[0][r];
                    e[(R + r) * 64] = rc[1][r];
                    e[(2 * R + r) * 64] = K[C - 1][r] * lp[C - 1][r];
                }
            }
            lds_barrier();
            if (edge) __builtin_amdgcn_s_setprio(3);
            {
                const ArgPtr<float> fpx = (ArgPtr<float>)fresh_args<ExArgs>()->fpx + x0;
                float rl1[R], rr1[R], rr2[R];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float *e = eR + lane;
                    rl1[r] = wave > 0 ? e[(((wave - 1) * 3 + 2) * R + r) * 64] : 0.0f;
                    rr1[r] = wave + 1 < W ? e[((wave + 1) * 3 * R + r) * 64] : 0.0f;
                    rr2[r] = wave + 1 < W ? e[(((wave + 1) * 3 + 1) * R + r) * 64] : 0.0f;
                }
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    if (c + 1 < C) fetch_v(c + 1);
                    const float fx = fpx[c];
                    if (c + 2 < C) {
#pragma unroll
                        for (int r = 0; r < R; ++r)
                            rc[c + (c + 2 < C ? 2 : 0)][r] = K[c + (c + 2 < C ? 2 : 0)][r] * lp[c + (c + 2 < C ? 2 : 0)][r];
                    }
                    const float d1 = dn1(rc[c][R - 1]), un1 = up1(rc[c][0]), un2 = up1(rc[c][1]);
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float xm = c >= 1 ? rc[c - (c >= 1)][r] : rl1[r];
                        const float xp = c + 1 < C ? rc[c + (c + 1 < C)][r] : rr1[r];
                        const float xq = c + 2 < C ? rc[c + (c + 2 < C ? 2 : 0)][r] : c + 2 == C ? rr1[r] : rr2[r];
                        const float zm = r >= 1 ? rc[c][r - (r >= 1)] : d1;
                        const float zp = r + 1 < R ? rc[c][r + (r + 1 < R)] : un1;
                        const float zq = r + 2 < R ? rc[c][r + (r + 2 < R ? 2 : 0)] : r + 2 == R ? un1 : un2;
                        const float dx = kC1 * (rc[c][r] - xp) + kC2 * (xm - xq);
                        const float dz = kC1 * (rc[c][r] - zp) + kC2 * (zm - zq);
                        lu[c][r] = cfu[c % 2][r] * lu[c][r] - dx;
                        lw[c][r] = cfw[c % 2][r] * lw[c][r] - dz;
                        lp[c][r] = fminf(fx, fpz[r]) * lp[c][r];
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        pin(lu[c][r]);
                        pin(lw[c][r]);
                        pin(lp[c][r]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // ---- exchange lu, hand out the next step's injection ----
            const bool exch = it > it0;
            if (exch) ++tag;
            constexpr int kMsg = kH * R * 64;
            u64 *box = nullptr;
            if (edge && exch) {
                const ArgPtr<ExArgs> k = fresh_args<ExArgs>();
                box = k->msg + ((size_t)(grp * k->c.P + j) * 2 + (tag & 1)) * (2 * kMsg) + voff / (4 * R);
                send_edges<R, C>(has_l, has_r, wave, W, box - 3 * kMsg, box + 4 * kMsg, tag, lu);
            }
            {
                float *f = sets + ((it - 1) & 1) * set_floats;
                if (i0.x >= 0) f[i0.x] = gn0;
                if (i1.x >= 0) f[i1.x] = gn1;
            }
            if (edge && exch)
                recv_edges<ExArgs, R, C>(has_l, has_r, wave, W, box, box + kMsg, tag, sh_place, dead, lu);
            if (edge) __builtin_amdgcn_s_setprio(0);
            put_q();
            lds_barrier();
        }
        // own columns out
        {
            const ArgPtr<ExArgs> k = fresh_args<ExArgs>();
            int x0 = x0w;
            unsigned voff = voff0;
            opaque_s(x0);
            opaque_v(voff);
            const int nxp = k->d.nxp, nzp = k->d.nzp, ld = k->d.ld, np = nxp * ld, fs = k->d.fs;
            const int zr = k->c.z0 + (int)(voff >> 2);
            const int os_ = window_os(k->c.W, C, j), oe_ = window_oe(k->c.W, C, j, k->c.P, nxp);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int x = x0 + c;
                if (x < os_ || x > oe_) continue;
                float *g = k->gk + (size_t)s * np + (size_t)(x - 1) * ld;
                const bool in_x = x >= 3 && x <= nxp - 2;
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (in_x && zr + r >= fs + 1 && zr + r <= nzp - 2) g[zr + r - 1] = gk[c][r];
                if (k->out) {
                    float *f = k->out + (size_t)s * 3 * np + (size_t)(x - 1) * ld;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (zr + r <= nzp) {
                            const unsigned o = zr + r - 1;
                            f[o] = lp[c][r];
                            f[np + o] = lu[c][r];
                            f[2 * np + o] = lw[c][r];
                        }
                }
            }
        }
        lds_barrier();               // the edges and the stages are rewritten by the next shot
    }
}

// Coefficients of a configuration, column by column (1 .. ncol, past nxp zero):
// {pressure update's, velocity updates', 1-kappa_p, 1-kappa_u, 1-kappa_w}[64 R rows from z0].
// The forward's pressure coefficient is K and its velocity coefficient B, the adjoint's the
// other way round.  They are zero outside the update regions: pressure rows zp0 .. nzp-2 and
// columns 3 .. nxp-2, velocity rows zv0 .. nzp-2 and columns 2 .. nxp-2 (the reference's
// regions hold one more row of u and one more column of w, whose stencils read only zeros:
// they stay zero).  Column 0 holds the factors of a column away from the side layers;
// fpx[x] is column x's 1-kappa_p on the interior rows.
__global__ void k_res_setup(Dims d, int R, int z0, int ncol, int zp0, int zv0, int adjoint,
                            const float2 *__restrict__ KB, const float2 *__restrict__ CP,
                            const float4 *__restrict__ CV, float *__restrict__ co, float *__restrict__ fpx) {
    const int row = blockIdx.x * blockDim.x + threadIdx.x, col = blockIdx.y;
    if (row >= 64 * R || col > ncol) return;
    const int z = z0 + row, x = col ? col : d.npml + 1;
    const bool in = z >= 1 && z <= d.nzp && x <= d.nxp;
    float K = 0.0f, B = 0.0f, fp = 1.0f, fu = 1.0f, fw = 1.0f;
    if (in) {
        const size_t k = pidx(d, z, x);
        const float2 kb = KB[k];
        const float4 cv = CV[k];
        K = kb.x;
        B = kb.y;
        fp = CP[k].y;
        fu = cv.y;
        fw = cv.z;
    }
    const bool rp = in && z >= zp0 && z <= d.nzp - 2 && x >= 3 && x <= d.nxp - 2;
    const bool rv = in && z >= zv0 && z <= d.nzp - 2 && x >= 2 && x <= d.nxp - 2;
    const size_t n = (size_t)64 * R;
    float *o = co + (size_t)col * 5 * n + row;
    o[0] = rp ? (adjoint ? B : K) : 0.0f;
    o[n] = rv ? (adjoint ? K : B) : 0.0f;
    o[2 * n] = fp;
    o[3 * n] = fu;
    o[4 * n] = fw;
    // the column's own damping: that of an interior row
    if (row == 0) fpx[col] = x <= d.nxp ? CP[pidx(d, d.npml + 1, x)].y : 1.0f;
}

// Start of a launch: the message words (tags) and the ticket counter.
__global__ void k_res_begin(u64 *__restrict__ msg, size_t n, Ctl *ctl, int clear_err) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        ctl->ticket = 0;
        if (clear_err) ctl->err = 0;
    }
    for (; i < n; i += (size_t)gridDim.x * blockDim.x) msg[i] = 0;
}

// What a forward of step kernels saves is whole.
__global__ void k_res_saved(Ctl *ctl, int saved) { ctl->bad[saved] = 0; }

// Receiver slots to traces: out[s][r][t] = in[s][t][map[s][r]], zero for a receiver past the
// shot's own count (map -1) and at t = 0; NaN everywhere if a wait of the job ran out, which
// also marks what it saved.  Tiles of 32 samples x 32 receivers through LDS; block (32, 8).
__global__ void k_res_traces(int nt, int ngmax, const int *__restrict__ map, const float *__restrict__ in,
                             float *__restrict__ out, Ctl *ctl, int saved) {
    __shared__ float tile[32][33];
    const int s = blockIdx.z, r0 = blockIdx.x * 32, t0 = blockIdx.y * 32;
    const bool bad = ctl->err != 0;
    if (saved >= 0 && blockIdx.x + blockIdx.y + blockIdx.z + threadIdx.x + threadIdx.y == 0) ctl->bad[saved] = bad;
    const int r = r0 + threadIdx.x;
    const int m = r < ngmax ? map[(size_t)s * ngmax + r] : -1;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int t = t0 + k;
        float v = 0.0f;
        if (m >= 0 && t < nt) v = in[((size_t)s * nt + t) * ngmax + m];
        tile[k][threadIdx.x] = bad ? __int_as_float(0x7fc00000) : v;
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int rr = r0 + k, t = t0 + threadIdx.x;
        if (rr < ngmax && t < nt) out[((size_t)s * ngmax + rr) * nt + t] = tile[threadIdx.x][k];
    }
}

}  // namespace rk
}  // namespace swit
