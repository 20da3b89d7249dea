// Smoother steps that ride on an operator launch, and how a launch finds the one meant for it.
//
// Plain C++ (the kernel that carries a step out is stencil_column_kernel).
#pragma once

namespace ppf
{
  /// What a smoother does with A x as stencil_column_kernel forms it, in place of storing it
  /// for a vector kernel to read back.
  enum class Smoother : int
  {
    None      = 0,
    Chebyshev = 1, ///< r = b - A x; d = c1 d + c2 r / diag (first: c2 r / diag); out = x + d
    Residual  = 2, ///< out = b - A x
    Dot       = 3  ///< out = A x, and per-workgroup partial sums of x . A x (CG)
  };

  /// Operands of a fused smoother step (one-field block vectors).  The inverse diagonal is
  /// the class table's entry where *ok, else the array (see chebyshev_table_kernel).
  template <typename ST>
  struct SmootherArgs
  {
    const ST  *b = nullptr;
    ST        *d = nullptr;
    const ST  *inv_diag = nullptr;
    const ST  *table = nullptr;
    const int *ok = nullptr;
    ST         c1 = ST(0), c2 = ST(0);
    int        first = 0;
    double    *partial = nullptr;
  };

  /// A smoother step waiting for the operator application dst = A src of a block that forms
  /// its A x.  It is there for that application only (SmootherScope) and no other launch
  /// takes it.
  template <typename T>
  struct SmootherRequest
  {
    int             block = -1;
    T              *dst   = nullptr;
    const T        *src   = nullptr;
    Smoother        kind  = Smoother::None;
    SmootherArgs<T> args {};
    bool            pending = false;
    bool            taken   = false;
    int             blocks  = 0; ///< workgroups of the launch that took it

    bool
    waits_for(int b, const T *to, const T *from) const
    {
      return pending && block == b && dst == to && src == from;
    }

    /// No launch is to carry the step out: the application gives A x.
    void
    withdraw()
    {
      pending = false;
    }

    /// A launch of n workgroups carries the step out.
    void
    take(int n)
    {
      pending = false;
      taken   = true;
      blocks  = n;
    }
  };

  /// Parks a request for the life of the object, which ends with the application however that
  /// ends (an exception leaves no request behind).
  template <typename T>
  struct SmootherScope
  {
    SmootherScope(SmootherRequest<T> &at, const SmootherRequest<T> &request)
      : slot(at)
    {
      slot         = request;
      slot.pending = true;
    }
    ~SmootherScope()
    {
      slot.pending = false;
    }
    SmootherScope(const SmootherScope &) = delete;
    SmootherScope &operator=(const SmootherScope &) = delete;
    SmootherRequest<T> &slot;
  };
} // namespace ppf
