// Stencil realization of operators on a 3-D vector field whose fluxes couple the
// components with constant coefficients (linear elasticity).
//
// A hook that submits, for each of three outputs c, the gradient term
//
//   t[c][d] = sum_{s,e} C[c][d][s][e] du_s/dx_e
//
// with constants C, no value term and the coupling of an orthotropic material assembles on
// the uniform GLL-collocated Q2 mesh to sums of tensor products of 1-D matrices, because the
// quadrature points are the nodes:
//
//   d = e: K_d (stiffness) times the lumped masses of the other axes;
//   d != e: G_d^T G_e times the lumped mass of the third axis, G = assembled (w_i D_ij).
//
// Divided by the lumped mass M_i of the node, and with h the cell edge,
//
//   L = K/m   even nodes (1, -8, 14, -8, 1), odd (0, -4, 8, -4, 0), in 1/h^2, with
//             mirrored values beyond a boundary (as in stencil_kernels.hpp);
//   G/m       even (1/2, -2, 0, 2, -1/2), odd (0, -1, 0, 1, 0), lower boundary
//             (0, 0, -3, 4, -1), upper boundary (1, -4, 3, 0, 0), in 1/h;
//   G^T/m     = -G/m + b, b = -6/h at a lower and +6/h at an upper boundary node, 0
//             elsewhere (integration by parts),
//
// so that, with g_d = G_d/m, the output at a node is M_i times
//
//   sum_s [ sum_d C[c][d][s][d] L_d u_s - sum_{d<e} (C[c][d][s][e] + C[c][e][s][d]) g_d g_e u_s
//           + sum_{d != e} C[c][d][s][e] b_d g_e u_s ].
//
// The reference evaluates the same operator cell by cell at the quadrature points
// (src/solvers/mf_operator.cc:17-80); only the order of the floating-point sums differs.
//
// Work decomposition: a workgroup owns a tile of tx columns by `strips` row pairs and
// marches over a chunk of z planes.  A thread owns one column of a row pair whose first
// row is even.  Per plane the three components are staged in shared memory with a halo of
// two nodes, corners included (loads of the next plane are in flight meanwhile, one
// barrier per plane); the thread reads a 5 x 5 neighbourhood per component for its two
// nodes, and its plane contributes forwards: a plane's values enter the running sums of
// the output planes within two of it, 5 planes x 3 components per row, where rings of
// u, g_x u and g_y u for a gather along z would take 45 values per row.
//
// The cell kernel this replaces for such operators (cell_column_kernel) evaluates the hook
// 27 times per cell, needs the whole register file of a SIMD for one wave and spills.
// Measured on linear elasticity, FP64: 64^3 Q2 cells 161 -> 45 us per application (103 MB of
// operands and results, 2.3 TB/s), 40 x 24 x 17 cells 33 -> 16 us.  What bounds it: 214
// registers, two waves per SIMD; per plane and wave 360 vector instructions, most of them
// FP64 (17 us of issue at 64^3), and 37 shared-memory instructions (13 us) that two waves
// do not fully overlap.  With 168 registers (three waves) it spills 56 of them.
#pragma once

#include "stencil_kernels.hpp"

namespace ppf
{
  constexpr int coupled_threads = 256;
  /// Staged positions per thread, component and plane: box <= 4 * 256 nodes.
  constexpr int coupled_loads = 4;

  /// Workgroups of the kernel a compute unit holds (registers).
  constexpr int coupled_resident = 2;

  /// The derivatives (d, e) of coefficient k (CoupledArgs::coef).
  constexpr int coupled_axes[12][2] = {{0, 0}, {1, 1}, {2, 2}, {0, 1}, {0, 2}, {1, 2},
                                       {0, 1}, {0, 2}, {1, 0}, {1, 2}, {2, 0}, {2, 1}};

  /// Whether coefficient k of operand s in output c can be nonzero for a material whose
  /// axes are the mesh's (isotropic, cubic, orthotropic): a direct derivative acts on its
  /// own component, a mixed one couples the two components of its axes.  Operators with
  /// any other coupling stay on the generic path: all 108 coefficients would not fit the
  /// scalar registers (tried: 358 of them spilled to vector lanes, 1.7 times the time).
  constexpr bool
  orthotropic_term(int k, int c, int s)
  {
    const int d = coupled_axes[k][0], e = coupled_axes[k][1];
    return d == e ? c == s : (c == d && s == e) || (c == e && s == d);
  }

  template <typename number>
  struct CoupledArgs
  {
    /// Coefficients of operand s in output c, coef[s][k][c]; k = 0 .. 5: the second
    /// derivatives xx, yy, zz, xy, xz, yz (the mixed ones carry the minus sign and both
    /// orders); k = 6 .. 11: C[c][d][s][e] of the boundary terms, (d, e) = xy, xz, yx, yz,
    /// zx, zy; all divided by the spacings.  Only the entries of orthotropic_term are read.
    number        coef[3][12][3];
    int           n[3], periodic[3];
    int           tx, strips; ///< tile: tx columns, 2 * strips rows
    int           tiles_x, tiles_y, chunks_z, z_chunk, n_blocks;
    const number *op[3];
    unsigned int  op_dmask[3]; ///< Dirichlet faces read as zero
    number       *dst[3];
    unsigned int  dst_dmask[3];
    unsigned int  any_dmask; ///< union of the masks
    int           keep_dirichlet; ///< Dirichlet nodes are left to dirichlet_faces_kernel
    /// Faces with a boundary term: not periodic and not Dirichlet for every output.
    unsigned int natural;
    number       sfac[3][3]; ///< output scale factors (StencilArgs::sfac)
    const int   *halt;
    int          nt_store;
  };

  /// Taps of g = G/m along one axis for offsets -2 .. 2, in 1/h.
  template <typename number>
  __device__ PPF_INLINE void
  derivative_taps(int i, int n, int periodic, number (&t)[5])
  {
    const bool lower = !periodic && i == 0, upper = !periodic && i == n - 1;
    const bool odd = (i & 1) != 0;
    t[0] = number(odd || lower ? 0.0 : (upper ? 1.0 : 0.5));
    t[1] = number(lower ? 0.0 : (upper ? -4.0 : (odd ? -1.0 : -2.0)));
    t[2] = number(lower ? -3.0 : (upper ? 3.0 : 0.0));
    t[3] = number(upper ? 0.0 : (lower ? 4.0 : (odd ? 1.0 : 2.0)));
    t[4] = number(odd || upper ? 0.0 : (lower ? -1.0 : -0.5));
  }

  template <typename number>
  __global__ void __launch_bounds__(coupled_threads, coupled_resident)
  coupled_stencil_kernel(const CoupledArgs<number> a)
  {
    extern __shared__ unsigned char coupled_shared[];
    number *lds = reinterpret_cast<number *>(coupled_shared);
    if (halted(a.halt))
      return;
    const int n0 = a.n[0], n1 = a.n[1], n2 = a.n[2];
    const int p0 = a.periodic[0], p1 = a.periodic[1], p2 = a.periodic[2];
    const int tid = threadIdx.x;

    // Consecutive tiles on one XCD (workgroups are dealt round-robin to the 8 XCDs).
    const int q8  = a.n_blocks / 8;
    const int b   = blockIdx.x;
    const int lb  = b < 8 * q8 ? (b % 8) * q8 + b / 8 : b;
    const int t_x = lb % a.tiles_x;
    const int t_r = lb / a.tiles_x;
    const int t_y = t_r % a.tiles_y;
    const int chk = t_r / a.tiles_y;
    const int x0 = t_x * a.tx, y0 = t_y * 2 * a.strips;
    const int zb = chk * a.z_chunk; // even (host)
    const int ze = min(zb + a.z_chunk, n2);

    const int          pitch = a.tx + 4;
    const int          box   = pitch * (2 * a.strips + 4);
    constexpr int      region = coupled_loads * coupled_threads;
    const unsigned int plane_bytes = unsigned(n0) * unsigned(n1) * unsigned(sizeof(number));
    buffer_rsrc        r_op[3], r_dst[3];
#pragma unroll
    for (int s = 0; s < 3; ++s)
      {
        r_op[s]  = make_rsrc(a.op[s]);
        r_dst[s] = make_rsrc(a.dst[s]);
      }

    // Staging positions of this thread.
    unsigned int st_off[coupled_loads], st_fb[coupled_loads];
#pragma unroll
    for (int k = 0; k < coupled_loads; ++k)
      {
        const int q  = min(tid + k * coupled_threads, box - 1);
        const int xs = source_coord(x0 - 2 + q % pitch, n0, p0);
        const int ys = source_coord(y0 - 2 + q / pitch, n1, p1);
        st_off[k]    = (unsigned(xs) + unsigned(n0) * unsigned(ys)) * unsigned(sizeof(number));
        st_fb[k]     = face_bits(xs, n0, p0, 0) | face_bits(ys, n1, p1, 1);
      }

    // Own column and row pair (threads beyond the tile shadow its first column).
    const bool active = tid < a.tx * a.strips;
    const int  tx     = active ? tid % a.tx : 0;
    const int  ts     = active ? tid / a.tx : 0;
    const int  x = x0 + tx, y = y0 + 2 * ts;
    const int  base = (2 * ts + 2) * pitch + tx + 2;
    bool       owned[2];
    owned[0] = active && x < n0 && y < n1;
    owned[1] = active && x < n0 && y + 1 < n1;
    const int    xc = min(x, n0 - 1), yc = min(y, n1 - 1);
    const bool   xodd = (xc & 1) != 0;
    const number wx0 = number(xodd ? 8.0 : 14.0), wx1 = number(xodd ? -4.0 : -8.0),
                 wx2 = number(xodd ? 0.0 : 1.0);
    number gx_t[5], gy_t[5]; // first row (even); the second row's are 0, -1, 0, 1, 0
    derivative_taps(xc, n0, p0, gx_t);
    derivative_taps(yc, n1, p1, gy_t);
    unsigned int own_fb[2], own_b[2];
    number       sxy[2];
    {
      const int    cx = scale_class<2>(xc, n0, p0);
      const number sx = cx == 0 ? a.sfac[0][0] : (cx == 1 ? a.sfac[0][1] : a.sfac[0][2]);
#pragma unroll
      for (int r = 0; r < 2; ++r)
        {
          const int    yr = min(y + r, n1 - 1);
          const int    cy = scale_class<2>(yr, n1, p1);
          const number sy = cy == 0 ? a.sfac[1][0] : (cy == 1 ? a.sfac[1][1] : a.sfac[1][2]);
          sxy[r]    = sx * sy;
          own_fb[r] = face_bits(xc, n0, p0, 0) | face_bits(yr, n1, p1, 1);
          own_b[r]  = (unsigned(xc) + unsigned(n0) * unsigned(yr)) * unsigned(sizeof(number));
        }
    }
    // Boundary terms of the x and y faces (b of this lane's column and first row).
    const bool   edge_xy = (a.natural & 0xfu) != 0 &&
                         (touches_face(x0, x0 + a.tx - 1, 0, n0, p0) ||
                          touches_face(y0, y0 + 2 * a.strips - 1, 0, n1, p1));
    const number bx = number(p0 ? 0.0 : (xc == 0 ? -6.0 : (xc == n0 - 1 ? 6.0 : 0.0)));
    const number by = number(p1 ? 0.0 : (yc == 0 ? -6.0 : (yc == n1 - 1 ? 6.0 : 0.0)));

    // Tiles whose box or chunk touches no face skip every Dirichlet test.
    const bool masked = (a.any_dmask & 0x3fu) != 0 &&
                        (touches_face(x0, x0 + a.tx - 1, 2, n0, p0) ||
                         touches_face(y0, y0 + 2 * a.strips - 1, 2, n1, p1) ||
                         touches_face(zb, ze - 1, 2, n2, p2));

    const auto source_z = [&](int z) {
      return unsigned(z) < unsigned(n2) ? z : source_coord(z, n2, p2);
    };
    number     pre[3][coupled_loads];
    const auto load = [&](int z) {
      const unsigned int po = unsigned(source_z(z)) * plane_bytes;
#pragma unroll
      for (int k = 0; k < coupled_loads; ++k)
        if (k * coupled_threads < box)
#pragma unroll
          for (int s = 0; s < 3; ++s)
            pre[s][k] = buffer_load<number>(r_op[s], st_off[k], po);
    };
    // Stages plane z (loaded before) and starts the loads of plane z + 1.  A component's
    // region holds every position a thread can store, so no lane is switched off.
    const auto stage = [&](int z, number *buf) {
      const unsigned int fbz = face_bits(source_z(z), n2, p2, 2);
#pragma unroll
      for (int k = 0; k < coupled_loads; ++k)
        if (k * coupled_threads < box)
          {
            if (masked)
#pragma unroll
              for (int s = 0; s < 3; ++s)
                pre[s][k] = ((st_fb[k] | fbz) & a.op_dmask[s]) ? number(0) : pre[s][k];
#pragma unroll
            for (int s = 0; s < 3; ++s)
              buf[s * region + tid + k * coupled_threads] = pre[s][k];
          }
      load(min(z + 1, ze + 1));
      __syncthreads();
    };

    // Running sums of output planes (slot k: plane zi - 2 + k of the pair iteration).
    number acc[5][3][2];
#pragma unroll
    for (int k = 0; k < 5; ++k)
#pragma unroll
      for (int c = 0; c < 3; ++c)
        acc[k][c][0] = acc[k][c][1] = number(0);

    // One plane: A = sum_s C_zz u (times the z taps of L), B = everything under g_z, and
    // the terms within the plane, added to `centre` when that output plane is owned.
    const auto plane_of = [&]<bool full>(std::bool_constant<full>, int z, const number *buf,
                                         number (&A)[3][2], number (&B)[3][2],
                                         number (&centre)[3][2]) {
      const bool edge_z  = full && !p2 && (z == 0 || z == n2 - 1) && (a.natural & 0x30u) != 0;
      const number bz    = number(z == 0 ? -6.0 : 6.0);
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int r = 0; r < 2; ++r)
          A[c][r] = B[c][r] = number(0);
#pragma unroll
      for (int s = 0; s < 3; ++s)
        {
          const auto term = [&](int k, int c, number value, number &sum) {
            if (orthotropic_term(k, c, s))
              sum = fma(a.coef[s][k][c], value, sum);
          };
          const bool    rows = full && s < 2; // g_x g_y u_s is used
          const number *v    = buf + s * region + base;
          number        u[5]; // own column, rows -2 .. 2
#pragma unroll
          for (int j = 0; j < 5; ++j)
            u[j] = v[(j - 2) * pitch];
          number gx[5], lx[2];
#pragma unroll
          for (int j = 0; j < 5; ++j)
            if (rows || j == 2 || j == 3)
              {
                const number *w   = v + (j - 2) * pitch;
                const number  xm2 = w[-2], xm1 = w[-1], xp1 = w[1], xp2 = w[2];
                gx[j] = fma(gx_t[0], xm2,
                            fma(gx_t[4], xp2,
                                fma(gx_t[1], xm1, fma(gx_t[3], xp1, gx_t[2] * u[j]))));
                if (j == 2 || j == 3)
                  lx[j - 2] = fma(wx2, xm2 + xp2, fma(wx1, xm1 + xp1, wx0 * u[j]));
              }
          number gy[2];
          gy[0] = fma(gy_t[0], u[0],
                      fma(gy_t[4], u[4], fma(gy_t[1], u[1], fma(gy_t[3], u[3], gy_t[2] * u[2]))));
          gy[1] = u[4] - u[2];
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int r = 0; r < 2; ++r)
              {
                term(2, c, u[2 + r], A[c][r]);
                term(4, c, gx[2 + r], B[c][r]);
                term(5, c, gy[r], B[c][r]);
              }
          if (full)
            {
              number ly[2];
              ly[0] = fma(number(14), u[2], fma(number(-8), u[1] + u[3], u[0] + u[4]));
              ly[1] = fma(number(8), u[3], number(-4) * (u[2] + u[4]));
#pragma unroll
              for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int r = 0; r < 2; ++r)
                  {
                    term(0, c, lx[r], centre[c][r]);
                    term(1, c, ly[r], centre[c][r]);
                  }
            }
          if (rows)
            {
              number gxy[2];
              gxy[0] = fma(gy_t[0], gx[0],
                           fma(gy_t[4], gx[4],
                               fma(gy_t[1], gx[1], fma(gy_t[3], gx[3], gy_t[2] * gx[2]))));
              gxy[1] = gx[4] - gx[2];
#pragma unroll
              for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int r = 0; r < 2; ++r)
                  term(3, c, gxy[r], centre[c][r]);
            }
          if (edge_xy)
            {
#pragma unroll
              for (int c = 0; c < 3; ++c)
                {
                  // only the first row of a pair can lie on a y face
                  term(7, c, bx * u[2], B[c][0]);
                  term(7, c, bx * u[3], B[c][1]);
                  term(9, c, by * u[2], B[c][0]);
                  if (full)
                    {
                      term(6, c, bx * gy[0], centre[c][0]);
                      term(6, c, bx * gy[1], centre[c][1]);
                      term(8, c, by * gx[2], centre[c][0]);
                    }
                }
            }
          if (edge_z)
            {
#pragma unroll
              for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int r = 0; r < 2; ++r)
                  {
                    term(10, c, bz * gx[2 + r], centre[c][r]);
                    term(11, c, bz * gy[r], centre[c][r]);
                  }
            }
        }
    };

    const auto plane = [&](int z, const number *buf, number (&A)[3][2], number (&B)[3][2],
                           number (&centre)[3][2]) {
      if (z >= zb && z < ze)
        plane_of(std::true_type {}, z, buf, A, B, centre);
      else
        plane_of(std::false_type {}, z, buf, A, B, centre);
    };

    const bool nt   = a.nt_store != 0;
    const auto emit = [&](int z, const number (&v)[3][2], number sz) {
      if (z < zb || z >= ze)
        return;
      const unsigned int zoff = unsigned(z) * plane_bytes;
      if (masked)
        {
          const unsigned int fbz = face_bits(z, n2, p2, 2);
#pragma unroll
          for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c)
              {
                const bool dir = ((own_fb[r] | fbz) & a.dst_dmask[c]) != 0;
                if (owned[r] && !(dir && a.keep_dirichlet))
                  buffer_store(dir ? number(0) : number(sxy[r] * sz * v[c][r]), r_dst[c],
                               own_b[r], zoff, nt);
              }
        }
      else
        {
#pragma unroll
          for (int r = 0; r < 2; ++r)
            if (owned[r])
#pragma unroll
              for (int c = 0; c < 3; ++c)
                buffer_store(number(sxy[r] * sz * v[c][r]), r_dst[c], own_b[r], zoff, nt);
        }
    };

    number *buf0 = lds, *buf1 = lds + 3 * region;
    number  A[3][2], B[3][2];
    load(zb - 2);
    for (int zi = zb - 2;; zi += 2)
      {
        // even plane zi: output planes zi - 2 .. zi + 2
        stage(zi, buf0);
        plane(zi, buf0, A, B, acc[2]);
        const bool   lo_c = !p2 && zi == 0, hi_c = !p2 && zi == n2 - 1;
        const bool   lo_p = !p2 && zi - 2 == 0, hi_p = !p2 && zi - 2 == n2 - 1;
        const bool   lo_n = !p2 && zi + 2 == 0, hi_n = !p2 && zi + 2 == n2 - 1;
        const number gp2 = number(lo_p ? -1.0 : (hi_p ? 0.0 : -0.5)); // output zi - 2
        const number g0  = number(lo_c ? -3.0 : (hi_c ? 3.0 : 0.0));  // output zi
        const number gm2 = number(lo_n ? 0.0 : (hi_n ? 1.0 : 0.5));   // output zi + 2
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            {
              const number av = A[c][r], bv = B[c][r];
              acc[0][c][r] += fma(gp2, bv, av);
              acc[1][c][r] += fma(number(-4), av, bv);
              acc[2][c][r] = fma(number(14), av, fma(g0, bv, acc[2][c][r]));
              acc[3][c][r] += fma(number(-4), av, -bv);
              acc[4][c][r] += fma(gm2, bv, av);
            }
        emit(zi - 2, acc[0], lo_p || hi_p ? a.sfac[2][2] : a.sfac[2][1]);
        emit(zi - 1, acc[1], a.sfac[2][0]);
        if (zi + 2 > ze + 1)
          break;
        // odd plane zi + 1: output planes zi .. zi + 2
        stage(zi + 1, buf1);
        plane(zi + 1, buf1, A, B, acc[3]);
        const number gp1 = number(lo_c ? 4.0 : (hi_c ? 0.0 : 2.0));   // output zi
        const number gm1 = number(lo_n ? 0.0 : (hi_n ? -4.0 : -2.0)); // output zi + 2
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            {
              const number av = A[c][r], bv = B[c][r];
              acc[0][c][r] = fma(number(-8), av, fma(gp1, bv, acc[2][c][r]));
              acc[1][c][r] = fma(number(8), av, acc[3][c][r]);
              acc[2][c][r] = fma(number(-8), av, fma(gm1, bv, acc[4][c][r]));
              acc[3][c][r] = number(0);
              acc[4][c][r] = number(0);
            }
      }
  }

  /// Diagonal of the same operator: M_i^scaling sum_d C[c][d][c][d] L_d(0).  (Mixed
  /// derivatives couple different components only, see orthotropic_term.)  Inverted as
  /// invert_diagonal_kernel does.
  template <typename number>
  __global__ void __launch_bounds__(block_size)
  coupled_inverse_diagonal_kernel(const GridDesc g, const CoupledArgs<number> a, int c,
                                  number *__restrict__ inv, int scaling)
  {
    const int64_t node = int64_t(blockIdx.x) * block_size + threadIdx.x;
    if (node >= g.n_nodes)
      return;
    int i[3];
    decompose<3>(g, node, g.nodes, i);
    if (is_dirichlet<3>(g, i, a.dst_dmask[c]))
      {
        inv[node] = number(1);
        return;
      }
    double k = 0.0;
    for (int d = 0; d < 3; ++d)
      k += double(a.coef[c][d][c]) * ((i[d] & 1) ? 8.0 : 14.0);
    const double v = node_scaling<3, 2>(g, i, scaling) * lumped_mass<3, 2>(g, i) * k;
    inv[node]      = number(v) == number(0) ? number(1) : number(1) / number(v);
  }
} // namespace ppf
