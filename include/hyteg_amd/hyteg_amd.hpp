// hyteg_amd.hpp -- C++ host API with HyTeG's Function / Operator / Solver
// shape, on top of the C ABI in hyteg_amd.h.  Header-only; solver control
// flow runs on the host, every numerical step is one or a few device kernels.
//
// Reference interfaces mirrored (paths relative to the HyTeG source tree):
//   PrimitiveStorage                    primitivestorage/PrimitiveStorage.hpp:116-220
//   P1Function<T>                       p1functionspace/P1Function.hpp:27, VertexDoFFunction.hpp:58-512
//   Operator<Src,Dst>::apply            operators/Operator.hpp:34-118
//   GSSmoothable / SORSmoothable        solvers/Smoothables.hpp:34-120
//   P1ConstantLaplaceOperator           constant_stencil_operator/P1ConstantOperator.hpp:167-168
//   P1toP1LinearRestriction/Prolongation gridtransferoperators/P1toP1Linear*.hpp
//   Solver<Op>                          solvers/Solver.hpp:27-34
//   GaussSeidelSmoother, SORSmoother    solvers/GaussSeidelSmoother.hpp:31-55, SORSmoother.hpp
//   CGSolver                            solvers/CGSolver.hpp:36-203
//   P2Function<T>                       p2functionspace/P2Function.hpp
//   P2ElementwiseOperator (div k grad)  elementwiseoperators/P2ElementwiseOperator.hpp:61-475
//   P2toP2Quadratic{Restriction,Prolongation} gridtransferoperators/P2toP2Quadratic*.cpp
//   ChebyshevSmoother, estimateRadius   solvers/ChebyshevSmoother.hpp:40-665
//   GeometricMultigridSolver            solvers/GeometricMultigridSolver.hpp:38-308
#pragma once

#include <cmath>
#include <functional>
#include <limits>
#include <memory>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <typeinfo>
#include <utility>
#include <vector>

#include "../hyteg_amd.h"

namespace hyteg_amd {

using uint_t = unsigned long;

enum DoFType : int
{
   None              = 0,
   Inner             = HG_INNER,
   DirichletBoundary = HG_DIRICHLET,
   NeumannBoundary   = HG_NEUMANN,
   FreeslipBoundary  = HG_FREESLIP,
   All               = HG_ALL
};
inline DoFType operator|( DoFType a, DoFType b )
{
   return DoFType( int( a ) | int( b ) );
}
enum UpdateType : int
{
   Replace = HG_REPLACE,
   Add     = HG_ADD
};
enum class CycleType
{
   VCYCLE,
   WCYCLE
};

// placeholder for "no projection" (operators/NoOperator.hpp)
struct NoOperator
{};

inline void check( hg_ctx* ctx, int status, const char* what )
{
   if ( status != HG_OK )
      throw std::runtime_error( std::string( what ) + ": " + hg_last_error( ctx ) );
}

// Owns an hg_ctx (one device, one stream).
class Context
{
 public:
   explicit Context( int device = 0 )
   {
      if ( hg_ctx_create( device, &ctx_ ) != HG_OK )
         throw std::runtime_error( "hg_ctx_create failed" );
   }
   ~Context()
   {
      if ( ctx_ )
         hg_ctx_destroy( ctx_ );
   }
   Context( const Context& )            = delete;
   Context& operator=( const Context& ) = delete;
   hg_ctx*  get() const { return ctx_; }
   void     synchronize() const { check( ctx_, hg_ctx_synchronize( ctx_ ), "synchronize" ); }

 private:
   hg_ctx* ctx_ = nullptr;
};

// PrimitiveStorage: macro mesh with boundary flags (setMeshBoundaryFlagsOnBoundary(1,0,true)).
class PrimitiveStorage
{
 public:
   PrimitiveStorage( std::shared_ptr< Context > ctx, hg_handle h )
   : owner_( std::move( ctx ) )
   , ctx_( owner_->get() )
   , h_( h )
   {}
   // view of a storage created elsewhere in the same context
   static std::shared_ptr< PrimitiveStorage > borrow( hg_ctx* ctx, hg_handle h )
   {
      return std::shared_ptr< PrimitiveStorage >( new PrimitiveStorage( ctx, h ) );
   }
   static std::shared_ptr< PrimitiveStorage >
       cuboid( std::shared_ptr< Context > ctx, const double lo[3], const double hi[3], int nx, int ny, int nz )
   {
      hg_handle h;
      check( ctx->get(), hg_storage_cuboid( ctx->get(), lo, hi, nx, ny, nz, &h ), "meshCuboid" );
      return std::make_shared< PrimitiveStorage >( ctx, h );
   }
   static std::shared_ptr< PrimitiveStorage >
       fromCells( std::shared_ptr< Context > ctx, const std::vector< double >& coords, const std::vector< int64_t >& cells )
   {
      hg_handle h;
      check( ctx->get(),
             hg_storage_create( ctx->get(), int( coords.size() / 3 ), coords.data(), int( cells.size() / 4 ), cells.data(), &h ),
             "storage" );
      return std::make_shared< PrimitiveStorage >( ctx, h );
   }
   hg_ctx*   ctx() const { return ctx_; }
   hg_handle handle() const { return h_; }

 private:
   PrimitiveStorage( hg_ctx* ctx, hg_handle h )
   : ctx_( ctx )
   , h_( h )
   {}
   std::shared_ptr< Context > owner_;
   hg_ctx*                    ctx_ = nullptr;
   hg_handle                  h_   = 0;
};

// FP16 storage tag: functions of this value type hold IEEE half values on the
// device; their scalars (assign coefficients, dot products) are float.
struct f16
{
   unsigned short bits;
};

template < typename T >
struct DTypeOf;
template <>
struct DTypeOf< double >
{
   static constexpr int value = HG_F64;
};
template <>
struct DTypeOf< float >
{
   static constexpr int value = HG_F32;
};
template <>
struct DTypeOf< f16 >
{
   static constexpr int value = HG_F16;
};
template < typename T >
struct ScalarOf
{
   using type = T;
};
template <>
struct ScalarOf< f16 >
{
   using type = float;
};

// P1Function<ValueType> (Space 1) and P2Function<ValueType> (Space 2): one
// device array per level; a P2 function of level L holds the values of the
// level-(L+1) vertex lattice (vertex DoFs at even, edge DoFs at odd points).
// Wraps an existing handle without owning it when constructed through `borrow`.
template < typename StorageType, int Space >
class LatticeFunction
{
 public:
   using valueType   = typename ScalarOf< StorageType >::type;
   using storageType = StorageType;
   using ValueType   = valueType;

   // nvec > 1: that many independent vectors interleaved per DoF
   LatticeFunction( const std::string& name, const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel,
                    uint_t maxLevel, int nvec = 1 )
   : name_( name )
   , storage_( storage )
   , ctx_( storage->ctx() )
   , owned_( true )
   , nvec_( nvec )
   {
      const int dt = DTypeOf< StorageType >::value;
      const int st = Space == 1 ? ( nvec == 1 ? hg_p1_function_create( ctx_, storage->handle(), int( minLevel ),
                                                                       int( maxLevel ), dt, &h_ ) :
                                                hg_p1_function_create_batched( ctx_, storage->handle(), int( minLevel ),
                                                                               int( maxLevel ), dt, nvec, &h_ ) ) :
                                  ( nvec == 1 ? hg_p2_function_create( ctx_, storage->handle(), int( minLevel ),
                                                                       int( maxLevel ), dt, &h_ ) :
                                                hg_p2_function_create_batched( ctx_, storage->handle(), int( minLevel ),
                                                                               int( maxLevel ), dt, nvec, &h_ ) );
      check( ctx_, st, Space == 1 ? "P1Function" : "P2Function" );
   }
   ~LatticeFunction()
   {
      if ( owned_ && h_ )
         hg_function_destroy( ctx_, h_ );
   }
   LatticeFunction( const LatticeFunction& )            = delete;
   LatticeFunction& operator=( const LatticeFunction& ) = delete;

   static std::unique_ptr< LatticeFunction > borrow( hg_ctx* ctx, hg_handle h )
   {
      return std::unique_ptr< LatticeFunction >( new LatticeFunction( ctx, h ) );
   }

   hg_handle handle() const { return h_; }
   hg_ctx*   ctx() const { return ctx_; }
   int       nvec() const { return nvec_; }
   // BoundaryCondition::createAllInnerBC (boundary/BoundaryConditions.cpp): every
   // DoF counts as Inner, so a flag selects all DoFs when it contains Inner and
   // none otherwise (the pressure of a Taylor-Hood function)
   void setAllInner( bool allInner = true ) { allInner_ = allInner; }
   bool isAllInner() const { return allInner_; }
   // per-vector dot products of interleaved functions
   std::vector< double > dotGlobalBatched( const LatticeFunction& other, uint_t level, DoFType flag = All ) const
   {
      std::vector< double > r( static_cast< size_t >( nvec_ ) );
      check( ctx_, hg_function_dot_batched( ctx_, h_, other.h_, int( level ), dofs( flag ), r.data() ),
             "dotGlobalBatched" );
      return r;
   }
   // vector k of this function = vector ksrc of other
   template < typename OtherT >
   void copyVector( int k, const LatticeFunction< OtherT, Space >& other, int ksrc, uint_t level ) const
   {
      check( ctx_, hg_function_copy_vector( ctx_, h_, k, other.handle(), ksrc, int( level ) ), "copyVector" );
   }
   // v_k *= scales[k] for every interleaved vector k
   void scaleBatched( const std::vector< double >& scales, uint_t level, DoFType flag = All ) const
   {
      if ( scales.size() != size_t( nvec_ ) )
         throw std::invalid_argument( "scaleBatched needs one scale per vector" );
      check( ctx_, hg_function_scale_batched( ctx_, h_, scales.data(), int( level ), dofs( flag ) ), "scaleBatched" );
   }

   void assign( const std::vector< ValueType >&                                            scalars,
                const std::vector< std::reference_wrapper< const LatticeFunction > >& functions,
                uint_t                                                                 level,
                DoFType                                                                flag = All ) const
   {
      linComb( scalars, functions, level, flag, false );
   }
   void add( const std::vector< ValueType >&                                            scalars,
             const std::vector< std::reference_wrapper< const LatticeFunction > >& functions,
             uint_t                                                                 level,
             DoFType                                                                flag = All ) const
   {
      linComb( scalars, functions, level, flag, true );
   }
   void interpolate( ValueType constant, uint_t level, DoFType flag = All ) const
   {
      check( ctx_, hg_function_interpolate_const( ctx_, h_, double( constant ), int( level ), dofs( flag ) ),
             "interpolate" );
   }
   // invertElementwise(level, flag): v = 1/v (zeros kept), FP64
   void invertElementwise( uint_t level, DoFType flag = All ) const
   {
      check( ctx_, hg_function_invert( ctx_, h_, int( level ), dofs( flag ) ), "invertElementwise" );
   }
   void setToZero( uint_t level ) const { interpolate( ValueType( 0 ), level, All ); }
   ValueType dotGlobal( const LatticeFunction& other, uint_t level, DoFType flag = All ) const
   {
      double r = 0.0;
      check( ctx_, hg_function_dot( ctx_, h_, other.h_, int( level ), dofs( flag ), &r ), "dotGlobal" );
      return ValueType( r );
   }
   // one fused Chebyshev step on this function (x): t = invDiag * (b - s) (b given)
   // or invDiag * s on flagged DoFs, 0 elsewhere; x += c t on flagged DoFs
   void chebyshevStep( const LatticeFunction& t, const LatticeFunction& s, const LatticeFunction* b,
                       const LatticeFunction& invDiag, double c, uint_t level, DoFType flag ) const
   {
      check( ctx_,
             hg_function_chebyshev_step( ctx_, h_, t.h_, s.h_, b ? b->h_ : 0, invDiag.h_, c, int( level ), dofs( flag ) ),
             "chebyshevStep" );
   }
   // the step with the step size of vector k in device slot slot0 + k
   void chebyshevStepSlots( const LatticeFunction& t, const LatticeFunction& s, const LatticeFunction* b,
                            const LatticeFunction& invDiag, int slot0, uint_t level, DoFType flag ) const
   {
      check( ctx_,
             hg_function_chebyshev_step_slots( ctx_, h_, t.h_, s.h_, b ? b->h_ : 0, invDiag.h_, slot0, int( level ),
                                               dofs( flag ) ),
             "chebyshevStepSlots" );
   }
   // dotGlobal into a device scalar slot of the context (no wait for the result)
   void dotToSlot( const LatticeFunction& other, uint_t level, DoFType flag, int slot ) const
   {
      check( ctx_, hg_function_dot_slot( ctx_, h_, other.h_, int( level ), dofs( flag ), slot ), "dotToSlot" );
   }
   // assign / add with scalars formed on the device: signs[i] * slot[num[i]] / slot[den[i]],
   // all zero while slot[gate] is nonzero (gate < 0: always formed)
   void linCombSlots( const std::vector< double >& signs, const std::vector< int >& num, const std::vector< int >& den,
                      const std::vector< std::reference_wrapper< const LatticeFunction > >& functions, uint_t level,
                      DoFType flag, bool add, int gate = -1 ) const
   {
      if ( signs.size() != functions.size() || num.size() != functions.size() || den.size() != functions.size() )
         throw std::invalid_argument( "linCombSlots needs one coefficient per function" );
      std::vector< hg_handle > hs;
      for ( const auto& f : functions )
         hs.push_back( f.get().h_ );
      check( ctx_,
             hg_function_lincomb_slots_gated( ctx_, h_, int( hs.size() ), signs.data(), num.data(), den.data(), hs.data(),
                                              int( level ), dofs( flag ), add ? 1 : 0, gate ),
             "linCombSlots" );
   }
   template < typename OtherT >
   void copyFrom( const LatticeFunction< OtherT, Space >& other, uint_t level ) const
   {
      check( ctx_, hg_function_copy_from( ctx_, h_, other.handle(), int( level ) ), "copyFrom" );
   }
   // multElementwise({a, b}, level, flag): this = a * b on flagged DoFs
   void multElementwise( const std::vector< std::reference_wrapper< const LatticeFunction > >& functions, uint_t level,
                         DoFType flag = All ) const
   {
      if ( functions.size() != 2 )
         throw std::invalid_argument( "multElementwise takes two functions" );
      check( ctx_,
             hg_function_mult( ctx_, h_, functions[0].get().h_, functions[1].get().h_, int( level ), dofs( flag ) ),
             "multElementwise" );
   }
   void communicate( uint_t level ) const { check( ctx_, hg_function_communicate( ctx_, h_, int( level ) ), "communicate" ); }

 private:
   LatticeFunction( hg_ctx* ctx, hg_handle h )
   : ctx_( ctx )
   , h_( h )
   , owned_( false )
   {
      check( ctx_, hg_function_nvec( ctx_, h_, &nvec_ ), "nvec" );
   }
   int dofs( DoFType flag ) const { return allInner_ ? ( ( flag & Inner ) ? int( All ) : 0 ) : int( flag ); }
   void linComb( const std::vector< ValueType >&                                            scalars,
                 const std::vector< std::reference_wrapper< const LatticeFunction > >& functions,
                 uint_t                                                                 level,
                 DoFType                                                                flagIn,
                 bool                                                                   add ) const
   {
      const int flag = dofs( flagIn );
      if ( scalars.size() != functions.size() )
         throw std::invalid_argument( "assign: sizes differ" );
      std::vector< double >    s( scalars.begin(), scalars.end() );
      std::vector< hg_handle > f;
      for ( const auto& r : functions )
         f.push_back( r.get().h_ );
      // the device kernel combines up to three sources per pass
      size_t i = 0;
      bool   first = true;
      do
      {
         const int n = int( std::min< size_t >( 3, f.size() - i ) );
         const int st =
             ( add || !first ) ? hg_function_add( ctx_, h_, n, s.data() + i, f.data() + i, int( level ), flag ) :
                                 hg_function_assign( ctx_, h_, n, s.data() + i, f.data() + i, int( level ), flag );
         check( ctx_, st, "assign" );
         i += size_t( n );
         first = false;
      } while ( i < f.size() );
   }

   std::string                         name_;
   std::shared_ptr< PrimitiveStorage > storage_;
   hg_ctx*                             ctx_   = nullptr;
   hg_handle                           h_        = 0;
   bool                                owned_    = true;
   int                                 nvec_     = 1;
   bool                                allInner_ = false;
};

// copyBCs(src, dst): dst takes src's boundary-condition mode (the solvers'
// temporaries follow the function they solve for, as copyBCs does in the
// reference's solvers); a no-op for composite functions
template < class F >
inline void copyBCs( const F&, F& )
{}
template < typename T, int S >
inline void copyBCs( const LatticeFunction< T, S >& src, LatticeFunction< T, S >& dst )
{
   dst.setAllInner( src.isAllInner() );
}

template < typename ValueType >
using P1Function = LatticeFunction< ValueType, 1 >;
template < typename ValueType >
using P2Function = LatticeFunction< ValueType, 2 >;

// Operator<Src,Dst>
template < class SrcT, class DstT >
class Operator
{
 public:
   using srcType = SrcT;
   using dstType = DstT;
   virtual ~Operator() = default;
   virtual void apply( const SrcT& src, const DstT& dst, uint_t level, DoFType flag, UpdateType updateType = Replace ) const = 0;
};

template < class F >
class GSSmoothable
{
 public:
   virtual ~GSSmoothable()                                                                    = default;
   virtual void smooth_gs( const F& dst, const F& rhs, uint_t level, DoFType flag ) const = 0;
};
template < class F >
class SORSmoothable
{
 public:
   virtual ~SORSmoothable() = default;
   virtual void smooth_sor( const F& dst, const F& rhs, typename F::valueType relax, uint_t level, DoFType flag ) const = 0;
};

// P1ConstantLaplaceOperator; VT is the value type of the functions it acts on
// (double, float, or f16 storage with FP32 arithmetic); one device operator
// serves every value type and any number of interleaved vectors
template < typename VT >
class P1ConstantLaplaceOperatorT : public Operator< P1Function< VT >, P1Function< VT > >,
                                   public GSSmoothable< P1Function< VT > >,
                                   public SORSmoothable< P1Function< VT > >
{
 public:
   P1ConstantLaplaceOperatorT( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel )
   : ctx_( storage->ctx() )
   , owned_( true )
   {
      check( ctx_, hg_p1_laplace_create( ctx_, storage->handle(), int( minLevel ), int( maxLevel ), &h_ ),
             "P1ConstantLaplaceOperator" );
   }
   static std::unique_ptr< P1ConstantLaplaceOperatorT > borrow( hg_ctx* ctx, hg_handle h )
   {
      return std::unique_ptr< P1ConstantLaplaceOperatorT >( new P1ConstantLaplaceOperatorT( ctx, h ) );
   }
   ~P1ConstantLaplaceOperatorT() override
   {
      if ( owned_ && h_ )
         hg_operator_destroy( ctx_, h_ );
   }
   void apply( const P1Function< VT >& src, const P1Function< VT >& dst, uint_t level, DoFType flag,
               UpdateType updateType = Replace ) const override
   {
      check( ctx_, hg_p1_apply( ctx_, h_, src.handle(), dst.handle(), int( level ), flag, updateType ), "apply" );
   }
   void smooth_gs( const P1Function< VT >& dst, const P1Function< VT >& rhs, uint_t level, DoFType flag ) const override
   {
      smooth_sor( dst, rhs, 1.0, level, flag );
   }
   void smooth_sor( const P1Function< VT >& dst, const P1Function< VT >& rhs, typename P1Function< VT >::valueType relax,
                    uint_t level, DoFType flag ) const override
   {
      check( ctx_, hg_p1_smooth_sor( ctx_, h_, dst.handle(), rhs.handle(), double( relax ), int( level ), flag ),
             "smooth_sor" );
   }
   hg_handle handle() const { return h_; }

 private:
   P1ConstantLaplaceOperatorT( hg_ctx* ctx, hg_handle h )
   : ctx_( ctx )
   , h_( h )
   , owned_( false )
   {}
   hg_ctx*   ctx_ = nullptr;
   hg_handle h_   = 0;
   bool      owned_;
};
using P1ConstantLaplaceOperator = P1ConstantLaplaceOperatorT< double >;

template < class F >
class RestrictionOperator
{
 public:
   virtual ~RestrictionOperator()                                                    = default;
   virtual void restrict( const F& function, uint_t sourceLevel, DoFType flag ) const = 0;
};
template < class F >
class ProlongationOperator
{
 public:
   virtual ~ProlongationOperator()                                                           = default;
   virtual void prolongate( const F& function, uint_t sourceLevel, DoFType flag ) const       = 0;
   virtual void prolongateAndAdd( const F& function, uint_t sourceLevel, DoFType flag ) const = 0;
};

template < typename ValueType = double >
class P1toP1LinearRestriction : public RestrictionOperator< P1Function< ValueType > >
{
 public:
   void restrict( const P1Function< ValueType >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      check( f.ctx(), hg_p1_restrict( f.ctx(), f.handle(), int( sourceLevel ), flag ), "restrict" );
   }
};
template < typename ValueType = double >
class P1toP1LinearProlongation : public ProlongationOperator< P1Function< ValueType > >
{
 public:
   void prolongate( const P1Function< ValueType >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      check( f.ctx(), hg_p1_prolongate( f.ctx(), f.handle(), int( sourceLevel ), flag, HG_REPLACE ), "prolongate" );
   }
   void prolongateAndAdd( const P1Function< ValueType >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      check( f.ctx(), hg_p1_prolongate( f.ctx(), f.handle(), int( sourceLevel ), flag, HG_ADD ), "prolongateAndAdd" );
   }
};

// OperatorWithInverseDiagonal<F> (solvers/Smoothables.hpp:96-120)
template < class F >
class OperatorWithInverseDiagonal
{
 public:
   virtual ~OperatorWithInverseDiagonal()                                = default;
   virtual std::shared_ptr< F > getInverseDiagonalValues() const          = 0;
   virtual void                 computeInverseDiagonalOperatorValues() = 0;
};

// P2ElementwiseOperator<p2_div_k_grad_blending_q4> with
// k(x) = exp(sum_m a_m sin(omega_m . x + phi_m))
// (elementwiseoperators/P2ElementwiseOperator.hpp:61-475)
//
// VT is the value type of the functions the operator acts on: double (FP64
// arithmetic), float or f16 (FP32 arithmetic, FP32 / FP16 storage of vectors
// and of the quadrature-point coefficients).  Operators of several value types
// may share one device operator (`borrow`).
template < typename VT >
class P2ElementwiseBlendingDivKGradOperatorT : public Operator< P2Function< VT >, P2Function< VT > >,
                                               public OperatorWithInverseDiagonal< P2Function< VT > >
{
 public:
   P2ElementwiseBlendingDivKGradOperatorT( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel,
                                           uint_t maxLevel, const std::vector< double >& a = {},
                                           const std::vector< double >& omega = {}, const std::vector< double >& phi = {} )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( true )
   {
      if ( omega.size() != 3 * a.size() || phi.size() != a.size() )
         throw std::invalid_argument( "k: omega needs 3 entries per mode, phi one" );
      check( ctx_,
             hg_p2_divkgrad_create( ctx_, storage->handle(), int( minLevel ), int( maxLevel ), int( a.size() ), a.data(),
                                    omega.data(), phi.data(), &h_ ),
             "P2ElementwiseBlendingDivKGradOperator" );
   }
   // batched form (no counterpart in the reference): nslot coefficient slots for
   // functions of nslot interleaved vectors, every slot k = 1 until
   // setSlotCoefficients gives it its own
   P2ElementwiseBlendingDivKGradOperatorT( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel,
                                           uint_t maxLevel, int nslot )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( true )
   , nslot_( nslot )
   {
      check( ctx_, hg_p2_divkgrad_create_batched( ctx_, storage->handle(), int( minLevel ), int( maxLevel ), nslot, &h_ ),
             "P2ElementwiseBlendingDivKGradOperator (batched)" );
   }
   // k of slot `slot` (same form as the constructor's); the stored tables and the
   // inverse diagonals of that slot are rebuilt
   void setSlotCoefficients( int slot, const std::vector< double >& a, const std::vector< double >& omega,
                             const std::vector< double >& phi )
   {
      if ( omega.size() != 3 * a.size() || phi.size() != a.size() )
         throw std::invalid_argument( "k: omega needs 3 entries per mode, phi one" );
      check( ctx_, hg_p2_divkgrad_set_slot( ctx_, h_, slot, int( a.size() ), a.data(), omega.data(), phi.data() ),
             "setSlotCoefficients" );
      if ( invDiag_ )
         for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
            check( ctx_, hg_p2_inverse_diagonal( ctx_, h_, int( L ), invDiag_->handle() ), "inverse diagonal" );
   }
   // an inactive slot is skipped by the apply (its result is zero): for slots
   // whose vectors are zero
   void setSlotActive( int slot, bool active )
   {
      check( ctx_, hg_p2_divkgrad_slot_active( ctx_, h_, slot, active ? 1 : 0 ), "setSlotActive" );
   }
   int slots() const { return nslot_; }
   static std::unique_ptr< P2ElementwiseBlendingDivKGradOperatorT >
       borrow( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h, uint_t minLevel, uint_t maxLevel )
   {
      return std::unique_ptr< P2ElementwiseBlendingDivKGradOperatorT >(
          new P2ElementwiseBlendingDivKGradOperatorT( storage, h, minLevel, maxLevel ) );
   }
   ~P2ElementwiseBlendingDivKGradOperatorT() override
   {
      if ( owned_ && h_ )
         hg_operator_destroy( ctx_, h_ );
   }
   void apply( const P2Function< VT >& src, const P2Function< VT >& dst, uint_t level, DoFType flag,
               UpdateType updateType = Replace ) const override
   {
      check( ctx_, hg_p2_apply( ctx_, h_, src.handle(), dst.handle(), int( level ), flag, updateType ), "apply" );
   }
   std::shared_ptr< P2Function< VT > > getInverseDiagonalValues() const override
   {
      if ( !invDiag_ )
         const_cast< P2ElementwiseBlendingDivKGradOperatorT* >( this )->computeInverseDiagonalOperatorValues();
      return invDiag_;
   }
   void computeInverseDiagonalOperatorValues() override
   {
      invDiag_ = std::make_shared< P2Function< VT > >( "inverseDiagonal", storage_, minLevel_, maxLevel_, nslot_ );
      for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
         check( ctx_, hg_p2_inverse_diagonal( ctx_, h_, int( L ), invDiag_->handle() ), "inverse diagonal" );
   }
   hg_handle handle() const { return h_; }
   uint_t    getMinLevel() const { return minLevel_; }
   uint_t    getMaxLevel() const { return maxLevel_; }
   const std::shared_ptr< PrimitiveStorage >& getStorage() const { return storage_; }

 private:
   P2ElementwiseBlendingDivKGradOperatorT( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h,
                                           uint_t minLevel, uint_t maxLevel )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , h_( h )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( false )
   {}
   std::shared_ptr< PrimitiveStorage >           storage_;
   hg_ctx*                                       ctx_ = nullptr;
   hg_handle                                     h_   = 0;
   uint_t                                        minLevel_, maxLevel_;
   bool                                          owned_;
   int                                           nslot_ = 1;
   std::shared_ptr< P2Function< VT > >           invDiag_;
};
using P2ElementwiseBlendingDivKGradOperator = P2ElementwiseBlendingDivKGradOperatorT< double >;

// P2toP2QuadraticRestriction / P2toP2QuadraticProlongation
// (gridtransferoperators/P2toP2QuadraticRestriction.cpp, P2toP2QuadraticProlongation.cpp)
template < typename ValueType = double >
class P2toP2QuadraticRestriction : public RestrictionOperator< P2Function< ValueType > >
{
 public:
   void restrict( const P2Function< ValueType >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      check( f.ctx(), hg_p2_restrict( f.ctx(), f.handle(), int( sourceLevel ), flag ), "restrict" );
   }
};
template < typename ValueType = double >
class P2toP2QuadraticProlongation : public ProlongationOperator< P2Function< ValueType > >
{
 public:
   void prolongate( const P2Function< ValueType >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      check( f.ctx(), hg_p2_prolongate( f.ctx(), f.handle(), int( sourceLevel ), flag, HG_REPLACE ), "prolongate" );
   }
   void prolongateAndAdd( const P2Function< ValueType >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      check( f.ctx(), hg_p2_prolongate( f.ctx(), f.handle(), int( sourceLevel ), flag, HG_ADD ), "prolongateAndAdd" );
   }
};

// Solver<Op>
// P2ConstantLaplaceOperator (constant_stencil_operator/P2ConstantOperator.hpp,
// P2ConstantOperator.cpp:100-1350): the P2 Laplacian of affine macro-cells with
// constant stencils, Gauss-Seidel / SOR smoothable, with inverse diagonal
class P2ConstantLaplaceOperator : public Operator< P2Function< double >, P2Function< double > >,
                                  public GSSmoothable< P2Function< double > >,
                                  public SORSmoothable< P2Function< double > >,
                                  public OperatorWithInverseDiagonal< P2Function< double > >
{
 public:
   P2ConstantLaplaceOperator( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( true )
   {
      check( ctx_, hg_p2_const_create( ctx_, storage->handle(), int( minLevel ), int( maxLevel ), &h_ ),
             "P2ConstantLaplaceOperator" );
   }
   static std::unique_ptr< P2ConstantLaplaceOperator >
       borrow( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h, uint_t minLevel, uint_t maxLevel )
   {
      return std::unique_ptr< P2ConstantLaplaceOperator >( new P2ConstantLaplaceOperator( storage, h, minLevel, maxLevel ) );
   }
   ~P2ConstantLaplaceOperator() override
   {
      if ( owned_ && h_ )
         hg_operator_destroy( ctx_, h_ );
   }
   void apply( const P2Function< double >& src, const P2Function< double >& dst, uint_t level, DoFType flag,
               UpdateType updateType = Replace ) const override
   {
      check( ctx_, hg_p2_const_apply( ctx_, h_, src.handle(), dst.handle(), int( level ), flag, updateType ),
             "P2ConstantLaplaceOperator::apply" );
   }
   void smooth_gs( const P2Function< double >& dst, const P2Function< double >& rhs, uint_t level,
                   DoFType flag ) const override
   {
      smooth_sor( dst, rhs, 1.0, level, flag );
   }
   void smooth_sor( const P2Function< double >& dst, const P2Function< double >& rhs, double relax, uint_t level,
                    DoFType flag ) const override
   {
      check( ctx_, hg_p2_const_smooth_sor( ctx_, h_, dst.handle(), rhs.handle(), int( level ), flag, relax ),
             "P2ConstantLaplaceOperator::smooth_sor" );
   }
   std::shared_ptr< P2Function< double > > getInverseDiagonalValues() const override
   {
      if ( !invDiag_ )
         const_cast< P2ConstantLaplaceOperator* >( this )->computeInverseDiagonalOperatorValues();
      return invDiag_;
   }
   void computeInverseDiagonalOperatorValues() override
   {
      invDiag_ = std::make_shared< P2Function< double > >( "inverseDiagonal", storage_, minLevel_, maxLevel_ );
      for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
         check( ctx_, hg_p2_const_inverse_diagonal( ctx_, h_, int( L ), invDiag_->handle() ), "inverse diagonal" );
   }
   hg_handle handle() const { return h_; }

 private:
   P2ConstantLaplaceOperator( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h, uint_t minLevel,
                              uint_t maxLevel )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , h_( h )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( false )
   {}
   std::shared_ptr< PrimitiveStorage >       storage_;
   hg_ctx*                                   ctx_;
   hg_handle                                 h_ = 0;
   uint_t                                    minLevel_, maxLevel_;
   bool                                      owned_;
   std::shared_ptr< P2Function< double > >   invDiag_;
};

template < class OperatorType >
class Solver
{
 public:
   virtual ~Solver() = default;
   virtual void solve( const OperatorType&                   A,
                       const typename OperatorType::srcType& x,
                       const typename OperatorType::dstType& b,
                       uint_t                                level ) = 0;
};

template < class OperatorType >
class GaussSeidelSmoother : public Solver< OperatorType >
{
 public:
   void solve( const OperatorType& A, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      if ( const auto* gs = dynamic_cast< const GSSmoothable< typename OperatorType::srcType >* >( &A ) )
         gs->smooth_gs( x, b, level, flag_ );
      else
         throw std::runtime_error( "The Gauss-Seidel Operator requires the GSSmoothable interface." );
   }

 private:
   DoFType flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

template < class OperatorType >
class SORSmoother : public Solver< OperatorType >
{
 public:
   explicit SORSmoother( double relax )
   : relax_( relax )
   {}
   void solve( const OperatorType& A, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      if ( const auto* s = dynamic_cast< const SORSmoothable< typename OperatorType::srcType >* >( &A ) )
         s->smooth_sor( x, b, relax_, level, flag_ );
      else
         throw std::runtime_error( "The SOR Operator requires the SORSmoothable interface." );
   }

 private:
   double  relax_;
   DoFType flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

template < class OperatorType >
class InverseDiagonalPreconditioner;

// CGSolver with the identity preconditioner (CGSolver.hpp:94-203, 340-358)
template < class OperatorType >
class CGSolver : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;
   using ValueType    = typename FunctionType::valueType;

   CGSolver( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel,
             uint_t maxIter = std::numeric_limits< uint_t >::max(), ValueType relativeTolerance = 1e-16,
             ValueType absoluteTolerance = 1e-16, std::shared_ptr< Solver< OperatorType > > preconditioner = nullptr )
   : maxIter_( maxIter )
   , relTol_( relativeTolerance )
   , absTol_( absoluteTolerance )
   , prec_( std::move( preconditioner ) )
   , p_( "p", storage, minLevel, maxLevel )
   , z_( "z", storage, minLevel, maxLevel )
   , ap_( "ap", storage, minLevel, maxLevel )
   , r_( "r", storage, minLevel, maxLevel )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   {
      if constexpr ( kDeviceScalars )
      {
         ctx_     = storage->ctx();
         storage_ = storage->handle();
         check( ctx_, hg_slots_alloc( ctx_, kSlotCount, &slot0_ ), "CGSolver slots" );
      }
   }
   ~CGSolver() override
   {
      if constexpr ( kDeviceScalars )
         hg_slots_free( ctx_, slot0_, kSlotCount );
   }
   CGSolver( const CGSolver& )            = delete;
   CGSolver& operator=( const CGSolver& ) = delete;

   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      if ( maxIter_ == 0 )
         return;
      if constexpr ( kDeviceScalars )
      {
         solveDeviceScalars( A, x, b, level );
         return;
      }
      copyBCs( x, p_ );
      copyBCs( x, z_ );
      copyBCs( x, ap_ );
      copyBCs( x, r_ );
      p_.setToZero( level );
      z_.setToZero( level );
      ap_.setToZero( level );
      r_.setToZero( level );
      A.apply( x, p_, level, flag_, Replace );
      r_.assign( { 1.0, -1.0 }, { b, p_ }, level, flag_ );
      precondition( A, level );
      p_.assign( { 1.0 }, { z_ }, level, flag_ );
      ValueType       prsold    = r_.dotGlobal( z_, level, flag_ );
      const ValueType res_start = std::sqrt( r_.dotGlobal( r_, level, flag_ ) );
      iterations_               = 0;
      if ( res_start < absTol_ )
         return;
      for ( uint_t i = 0; i < maxIter_; ++i )
      {
         A.apply( p_, ap_, level, flag_, Replace );
         const ValueType pAp   = p_.dotGlobal( ap_, level, flag_ );
         const ValueType alpha = prsold / pAp;
         x.add( { alpha }, { p_ }, level, flag_ );
         r_.add( { -alpha }, { ap_ }, level, flag_ );
         const ValueType rsnew  = r_.dotGlobal( r_, level, flag_ );
         const ValueType relRes = std::sqrt( rsnew ) / res_start;
         iterations_            = i;
         if ( relRes < relTol_ || std::sqrt( rsnew ) < absTol_ )
            break;
         z_.interpolate( ValueType( 0 ), level, All );
         precondition( A, level );
         const ValueType prsnew = r_.dotGlobal( z_, level, flag_ );
         const ValueType beta   = prsnew / prsold;
         p_.assign( { 1.0, beta }, { z_, p_ }, level, flag_ );
         prsold = prsnew;
      }
   }
   uint_t getIterations() const { return iterations_; }
   // exactly maxIter iterations with no residual read back (no host
   // synchronisation, so a surrounding V-cycle can be captured into a HIP graph):
   // the stopping test runs on the device and, once it holds, zeroes the step
   // sizes of the remaining iterations, so the iterate is the one the host-tested
   // loop returns; FP64 lattice functions only
   void setFixedIterations( bool fixed )
   {
      if ( fixed && !kDeviceScalars )
         throw std::invalid_argument( "fixed-iteration CG needs FP64 lattice functions" );
      fixed_ = fixed;
   }

 private:
   // FP64 lattice functions keep pAp, r.r and r.z in device slots of the context
   static constexpr bool kDeviceScalars =
       std::is_same_v< FunctionType, LatticeFunction< double, 1 > > || std::is_same_v< FunctionType, LatticeFunction< double, 2 > >;
   // slots: r.r, pAp, r.z (two, alternating), r0.r0 and the converged flag
   static constexpr int kSlotCount = 6;

   // The iteration above with its scalars on the device: alpha = r.z / pAp and
   // beta = r.z_new / r.z are formed inside the update kernels from slot values,
   // and r.r is the one value read back per iteration (for the stopping test), so
   // the iterates and the stopping step are those of the host-scalar loop.
   void solveDeviceScalars( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level )
   {
      // the P2 diffusion operator solves its small levels in one launch
      if constexpr ( std::is_same_v< OperatorType, P2ElementwiseBlendingDivKGradOperatorT< double > > )
      {
         // its DoF types are the mesh's: not for an x that counts every DoF as Inner; its
         // operator and preconditioner are these classes themselves, not derived ones
         const Solver< OperatorType >* prec = prec_.get();
         const bool jacobi = prec && typeid( *prec ) == typeid( InverseDiagonalPreconditioner< OperatorType > );
         if ( !fixed_ && !x.isAllInner() && typeid( A ) == typeid( OperatorType ) && ( !prec || jacobi ) &&
              workspaceFits( x, level ) )
         {
            int its = 0, applied = 0;
            check( ctx_,
                   hg_p2_cg_assembled( ctx_, A.handle(), x.handle(), b.handle(), int( level ), int( flag_ ),
                                       int( std::min< uint_t >( maxIter_, uint_t( std::numeric_limits< int >::max() ) ) ),
                                       relTol_, absTol_, jacobi ? 1 : 0, &its, &applied ),
                   "CGSolver" );
            if ( applied )
            {
               // left behind as by the loop: a solve captured later cannot allocate it
               if ( jacobi )
                  A.getInverseDiagonalValues();
               iterations_ = uint_t( its );
               return;
            }
         }
      }
      const int rr = slot0_, pap = slot0_ + 1, rr0 = slot0_ + 4, done = slot0_ + 5;
      int       rz[2] = { slot0_ + 2, slot0_ + 3 }, cur = 0;
      copyBCs( x, p_ );
      copyBCs( x, z_ );
      copyBCs( x, ap_ );
      copyBCs( x, r_ );
      p_.setToZero( level );
      z_.setToZero( level );
      ap_.setToZero( level );
      r_.setToZero( level );
      A.apply( x, p_, level, flag_, Replace );
      r_.assign( { 1.0, -1.0 }, { b, p_ }, level, flag_ );
      precondition( A, level );
      p_.assign( { 1.0 }, { z_ }, level, flag_ );
      r_.dotToSlot( z_, level, flag_, rz[cur] );
      double res_start = 0.0;
      iterations_      = 0;
      const int gate   = fixed_ ? done : -1;
      if ( !fixed_ )
      {
         r_.dotToSlot( r_, level, flag_, rr );
         check( ctx_, hg_slots_read( ctx_, rr, 1, &res_start ), "CGSolver" );
         res_start = std::sqrt( res_start );
         if ( res_start < absTol_ )
            return;
      }
      else
      {
         r_.dotToSlot( r_, level, flag_, rr0 );
         check( ctx_, hg_slots_cg_stop( ctx_, rr, rr0, relTol_, absTol_, done, 1 ), "CGSolver" );
      }
      for ( uint_t i = 0; i < maxIter_; ++i )
      {
         A.apply( p_, ap_, level, flag_, Replace );
         p_.dotToSlot( ap_, level, flag_, pap );
         x.linCombSlots( { 1.0 }, { rz[cur] }, { pap }, { p_ }, level, flag_, true, gate );
         r_.linCombSlots( { -1.0 }, { rz[cur] }, { pap }, { ap_ }, level, flag_, true, gate );
         iterations_ = i;
         if ( !fixed_ )
         {
            r_.dotToSlot( r_, level, flag_, rr );
            double rsnew = 0.0;
            check( ctx_, hg_slots_read( ctx_, rr, 1, &rsnew ), "CGSolver" );
            const double relRes = std::sqrt( rsnew ) / res_start;
            if ( relRes < relTol_ || std::sqrt( rsnew ) < absTol_ )
               break;
         }
         else
         {
            if ( i + 1 == maxIter_ )
               break;
            r_.dotToSlot( r_, level, flag_, rr );
            check( ctx_, hg_slots_cg_stop( ctx_, rr, rr0, relTol_, absTol_, done, 0 ), "CGSolver" );
         }
         z_.interpolate( 0.0, level, All );
         precondition( A, level );
         r_.dotToSlot( z_, level, flag_, rz[1 - cur] );
         p_.linCombSlots( { 1.0, 1.0 }, { -1, rz[1 - cur] }, { -1, rz[cur] }, { z_, p_ }, level, flag_, false, gate );
         cur = 1 - cur;
      }
   }

   // whether p, z, ap and r hold the level and live on x's storage (the loop fails
   // where they do not)
   bool workspaceFits( const FunctionType& x, uint_t level ) const
   {
      hg_handle s = 0;
      check( ctx_, hg_function_storage( ctx_, x.handle(), &s ), "CGSolver" );
      return s == storage_ && level >= minLevel_ && level <= maxLevel_;
   }

   // z = M^-1 r (identity when no preconditioner is given)
   void precondition( const OperatorType& A, uint_t level )
   {
      if ( prec_ )
         prec_->solve( A, z_, r_, level );
      else
         z_.assign( { 1.0 }, { r_ }, level, flag_ );
   }
   uint_t                                    maxIter_;
   ValueType                                 relTol_, absTol_;
   std::shared_ptr< Solver< OperatorType > > prec_;
   FunctionType                              p_, z_, ap_, r_;
   uint_t                                    minLevel_, maxLevel_;
   DoFType                                   flag_       = Inner | NeumannBoundary | FreeslipBoundary;
   uint_t                                    iterations_ = 0;
   hg_ctx*                                   ctx_        = nullptr;
   hg_handle                                 storage_    = 0;
   int                                       slot0_      = -1;
   bool                                      fixed_      = false;
};

// Preconditioner z = D^-1 r with the operator's inverse diagonal
// (ApplyPreconditioner over ApplyFunctionMultiplicationWrapper,
// solvers/SubstitutePreconditioner.hpp:120-158)
template < class OperatorType >
class InverseDiagonalPreconditioner : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;
   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      const auto* withDiag = dynamic_cast< const OperatorWithInverseDiagonal< FunctionType >* >( &A );
      if ( !withDiag )
         throw std::runtime_error( "the preconditioner requires the OperatorWithInverseDiagonal interface" );
      x.multElementwise( { *withDiag->getInverseDiagonalValues(), b }, level, flag_ );
   }

 private:
   DoFType flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

// ChebyshevSmoother (solvers/ChebyshevSmoother.hpp:40-420): x += p(D^-1 A) D^-1 (b - A x)
// with the polynomial p of degree order-1 for which
// 1 - t p(t) = T_order((theta - t)/delta) / T_order(theta/delta) on [lower, upper].
//
// With a projection (ChebyshevSmoother<Op, P2ProjectNormalOperator>), every
// preconditioned correction D^-1 r is projected on the projectionFlag DoFs before
// it is added to x (ChebyshevSmoother.hpp:186-231).
template < class F >
struct IsLatticeFunction : std::false_type
{};
template < class T, int Space >
struct IsLatticeFunction< LatticeFunction< T, Space > > : std::true_type
{};

template < class OperatorType, class ProjectionOperatorType = NoOperator >
class ChebyshevSmoother : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;
   using ValueType    = typename FunctionType::valueType;
   // scalar lattice functions run each step as one fused pass
   static constexpr bool kFusedSteps = IsLatticeFunction< FunctionType >::value;

   ChebyshevSmoother( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel )
   : ChebyshevSmoother( storage, minLevel, maxLevel, 1 )
   {}
   // temporaries of nvec interleaved vectors (multi-vector functions)
   ChebyshevSmoother( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel, int nvec )
   : minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , coefficients_( maxLevel - minLevel + 1 )
   , tmp1_( "cheby_tmp1", storage, minLevel, maxLevel, nvec )
   , tmp2_( "cheby_tmp2", storage, minLevel, maxLevel, nvec )
   {}
   // (storage, minLevel, maxLevel, lowMemoryMode, projection, projectionFlag); the
   // temporaries are always kept (lowMemoryMode only selects where they live there)
   ChebyshevSmoother( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel,
                      bool /* lowMemoryMode */, std::shared_ptr< ProjectionOperatorType > projection,
                      DoFType projectionFlag = FreeslipBoundary )
   : ChebyshevSmoother( storage, minLevel, maxLevel )
   {
      projection_     = std::move( projection );
      projectionFlag_ = projectionFlag;
   }

   // setupCoefficients(order, spectralRadius, upperFactor, lowerFactor)
   void setupCoefficients( uint_t order, double spectralRadius, double upperFactor = 1.2, double lowerFactor = 0.3 )
   {
      for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
         coefficients_[L - minLevel_] = coefficientsFor( order, lowerFactor * spectralRadius, upperFactor * spectralRadius );
   }
   void setupCoefficientsOnLevel( uint_t order, double spectralRadius, uint_t level, double upperFactor = 1.2,
                                  double lowerFactor = 0.3 )
   {
      coefficients_.at( level - minLevel_ ) =
          coefficientsFor( order, lowerFactor * spectralRadius, upperFactor * spectralRadius );
   }
   const std::vector< double >& coefficients( uint_t level ) const { return coefficients_.at( level - minLevel_ ); }

   // interleaved multi-vector functions (no counterpart in the reference): vector
   // k gets the coefficients of spectralRadius[k] on every level.  They live in
   // device slots of the context (order x nvec), so a V-cycle captured into a
   // graph takes new values written between its launches.
   void setupCoefficientsPerVector( uint_t order, const std::vector< double >& spectralRadius, hg_ctx* ctx,
                                    double upperFactor = 1.2, double lowerFactor = 0.3 )
   {
      const int nv = int( spectralRadius.size() );
      if ( vecSlot0_ < 0 )
      {
         check( ctx, hg_slots_alloc( ctx, int( order ) * nv, &vecSlot0_ ), "Chebyshev slots" );
         vecCtx_ = ctx;
         vecN_   = nv;
         vecOrd_ = order;
      }
      if ( nv != vecN_ || order != vecOrd_ )
         throw std::invalid_argument( "per-vector Chebyshev coefficients: order and vector count are fixed" );
      std::vector< double > v( size_t( order ) * size_t( nv ) );
      for ( int k = 0; k < nv; ++k )
      {
         const std::vector< double > c = coefficientsFor( order, lowerFactor * spectralRadius[size_t( k )],
                                                          upperFactor * spectralRadius[size_t( k )] );
         for ( uint_t i = 0; i < order; ++i )
            v[size_t( i ) * size_t( nv ) + size_t( k )] = c[i];
      }
      check( ctx, hg_slots_write( ctx, vecSlot0_, int( v.size() ), v.data() ), "Chebyshev slots" );
   }
   ~ChebyshevSmoother() override
   {
      if ( vecSlot0_ >= 0 )
         hg_slots_free( vecCtx_, vecSlot0_, int( vecOrd_ ) * vecN_ );
   }

   // monomial coefficients of p from the Chebyshev recurrence T_{j+1} = 2 s T_j - T_{j-1}
   // in s = (theta - t) / delta
   static std::vector< double > coefficientsFor( uint_t order, double lower, double upper )
   {
      if ( order < 1 || order > 16 )
         throw std::invalid_argument( "Chebyshev order must be 1..16" );
      const double          theta = 0.5 * ( upper + lower ), delta = 0.5 * ( upper - lower );
      const double          a = theta / delta, b = -1.0 / delta;
      std::vector< double > prev( order + 2, 0.0 ), cur( order + 2, 0.0 ), next( order + 2, 0.0 );
      prev[0] = 1.0;
      cur[0]  = a;
      cur[1]  = b;
      for ( uint_t j = 1; j < order; ++j )
      {
         for ( uint_t i = 0; i <= j + 1; ++i )
            next[i] = 2.0 * ( a * cur[i] + ( i > 0 ? b * cur[i - 1] : 0.0 ) ) - prev[i];
         prev = cur;
         cur  = next;
      }
      std::vector< double > c( order );
      for ( uint_t i = 0; i < order; ++i )
         c[i] = -cur[i + 1] / cur[0];
      return c;
   }

   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      const auto* withDiag = dynamic_cast< const OperatorWithInverseDiagonal< FunctionType >* >( &A );
      if ( !withDiag )
         throw std::runtime_error( "The Chebyshev-Smoother requires the OperatorWithInverseDiagonal interface." );
      const auto& invDiag = *withDiag->getInverseDiagonalValues();
      if constexpr ( kFusedSteps )
      {
         if ( vecSlot0_ >= 0 )
         {
            if ( x.nvec() != vecN_ || projection_ )
               throw std::runtime_error( "per-vector Chebyshev coefficients: vector count mismatch or projection" );
            A.apply( x, tmp2_, level, flag_ );
            x.chebyshevStepSlots( tmp1_, tmp2_, &b, invDiag, vecSlot0_, level, flag_ );
            for ( uint_t k = 1; k < vecOrd_; ++k )
            {
               A.apply( tmp1_, tmp2_, level, flag_ );
               x.chebyshevStepSlots( tmp1_, tmp2_, nullptr, invDiag, vecSlot0_ + int( k ) * vecN_, level, flag_ );
            }
            return;
         }
      }
      const std::vector< double >& c = coefficients_.at( level - minLevel_ );
      if ( c.empty() )
         throw std::runtime_error( "Chebyshev coefficients are not set up" );
      A.apply( x, tmp2_, level, flag_ );
      if constexpr ( kFusedSteps )
      {
         // without a projection each step is one pass over the DoFs (same values)
         if ( !projection_ )
         {
            x.chebyshevStep( tmp1_, tmp2_, &b, invDiag, double( ValueType( c[0] ) ), level, flag_ );
            for ( size_t k = 1; k < c.size(); ++k )
            {
               A.apply( tmp1_, tmp2_, level, flag_ );
               x.chebyshevStep( tmp1_, tmp2_, nullptr, invDiag, double( ValueType( c[k] ) ), level, flag_ );
            }
            return;
         }
      }
      tmp2_.assign( { 1.0, -1.0 }, { b, tmp2_ }, level, flag_ );
      tmp1_.setToZero( level );
      tmp1_.multElementwise( { invDiag, tmp2_ }, level, flag_ );
      project( level );
      x.add( { ValueType( c[0] ) }, { tmp1_ }, level, flag_ );
      for ( size_t k = 1; k < c.size(); ++k )
      {
         A.apply( tmp1_, tmp2_, level, flag_ );
         tmp1_.setToZero( level );
         tmp1_.multElementwise( { invDiag, tmp2_ }, level, flag_ );
         project( level );
         x.add( { ValueType( c[k] ) }, { tmp1_ }, level, flag_ );
      }
   }

 private:
   void project( uint_t level ) const
   {
      if constexpr ( !std::is_same< ProjectionOperatorType, NoOperator >::value )
         if ( projection_ )
            projection_->project( tmp1_, level, projectionFlag_ );
   }
   uint_t                                    minLevel_, maxLevel_;
   std::vector< std::vector< double > >      coefficients_;
   FunctionType                              tmp1_, tmp2_;
   int                                       vecSlot0_ = -1, vecN_ = 0;
   uint_t                                    vecOrd_   = 0;
   hg_ctx*                                   vecCtx_   = nullptr;
   DoFType                                   flag_ = Inner | NeumannBoundary | FreeslipBoundary;
   std::shared_ptr< ProjectionOperatorType > projection_;
   DoFType                                   projectionFlag_ = FreeslipBoundary;
};

// Coarse "solver" made of a fixed number of smoother sweeps (used for
// interleaved multi-vector hierarchies, whose CG would need per-vector scalars)
template < class OperatorType >
class SmootherSweeps : public Solver< OperatorType >
{
 public:
   SmootherSweeps( std::shared_ptr< Solver< OperatorType > > smoother, uint_t sweeps )
   : smoother_( std::move( smoother ) )
   , sweeps_( sweeps )
   {}
   void solve( const OperatorType& A, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      for ( uint_t i = 0; i < sweeps_; ++i )
         smoother_->solve( A, x, b, level );
   }

 private:
   std::shared_ptr< Solver< OperatorType > > smoother_;
   uint_t                                    sweeps_;
};

namespace chebyshev {
// estimateRadius (ChebyshevSmoother.hpp:656-665): power iteration on D^-1 A with
// flag All (numerictools/SpectrumEstimation.hpp:56-90); x is the start vector and
// holds the last iterate on return
template < class OperatorType >
double estimateRadius( const OperatorType& A, uint_t level, uint_t maxIter, const typename OperatorType::srcType& x,
                       const typename OperatorType::srcType& tmp )
{
   using FunctionType   = typename OperatorType::srcType;
   const auto* withDiag = dynamic_cast< const OperatorWithInverseDiagonal< FunctionType >* >( &A );
   if ( !withDiag )
      throw std::runtime_error( "estimateRadius requires the OperatorWithInverseDiagonal interface" );
   const auto& invDiag = *withDiag->getInverseDiagonalValues();
   auto        applyDA = [&]( const FunctionType& src, const FunctionType& dst ) {
      A.apply( src, dst, level, All );
      dst.multElementwise( { invDiag, dst }, level, All );
   };
   double norm = std::sqrt( double( x.dotGlobal( x, level, All ) ) );
   x.assign( { 1.0 / norm }, { x }, level, All );
   applyDA( x, tmp );
   double radius = 0.0;
   for ( uint_t it = 1; it <= maxIter; ++it )
   {
      norm = std::sqrt( double( tmp.dotGlobal( tmp, level, All ) ) );
      x.assign( { 1.0 / norm }, { tmp }, level, All );
      applyDA( x, tmp );
      radius = double( x.dotGlobal( tmp, level, All ) );
   }
   return radius;
}
// estimateRadius for each vector of an interleaved multi-vector function (no
// counterpart in the reference): the same power iteration with per-vector norms
// and Rayleigh quotients; a zero start vector gives radius 0
template < class OperatorType >
std::vector< double > estimateRadiusPerVector( const OperatorType& A, uint_t level, uint_t maxIter,
                                               const typename OperatorType::srcType& x,
                                               const typename OperatorType::srcType& tmp )
{
   using FunctionType   = typename OperatorType::srcType;
   const auto* withDiag = dynamic_cast< const OperatorWithInverseDiagonal< FunctionType >* >( &A );
   if ( !withDiag )
      throw std::runtime_error( "estimateRadius requires the OperatorWithInverseDiagonal interface" );
   const auto& invDiag = *withDiag->getInverseDiagonalValues();
   auto        applyDA = [&]( const FunctionType& src, const FunctionType& dst ) {
      A.apply( src, dst, level, All );
      dst.multElementwise( { invDiag, dst }, level, All );
   };
   auto inverseNorms = []( std::vector< double > nn ) {
      for ( double& v : nn )
         v = v > 0.0 ? 1.0 / std::sqrt( v ) : 1.0;
      return nn;
   };
   x.scaleBatched( inverseNorms( x.dotGlobalBatched( x, level, All ) ), level, All );
   applyDA( x, tmp );
   std::vector< double > radius( static_cast< size_t >( x.nvec() ), 0.0 );
   for ( uint_t it = 1; it <= maxIter; ++it )
   {
      const std::vector< double > inv = inverseNorms( tmp.dotGlobalBatched( tmp, level, All ) );
      x.assign( { 1.0 }, { tmp }, level, All );
      x.scaleBatched( inv, level, All );
      applyDA( x, tmp );
      radius = x.dotGlobalBatched( tmp, level, All );
   }
   return radius;
}
} // namespace chebyshev

// Coarse solver of a reduced-precision multigrid hierarchy that solves in FP64:
// b is cast up, `solver` (e.g. PCG to 1e-14) runs on the FP64 operator, and the
// result is cast back.
template < class OperatorType, class OperatorType64 >
class FP64CoarseSolver : public Solver< OperatorType >
{
 public:
   using FunctionType   = typename OperatorType::srcType;
   using FunctionType64 = typename OperatorType64::srcType;
   FP64CoarseSolver( const std::shared_ptr< PrimitiveStorage >& storage, uint_t level, const OperatorType64& A64,
                     std::shared_ptr< Solver< OperatorType64 > > solver )
   : A64_( A64 )
   , solver_( std::move( solver ) )
   , x64_( "coarse_x64", storage, level, level )
   , b64_( "coarse_b64", storage, level, level )
   {}
   void solve( const OperatorType&, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      b64_.copyFrom( b, level );
      x64_.setToZero( level );
      solver_->solve( A64_, x64_, b64_, level );
      x.copyFrom( x64_, level );
   }

 private:
   const OperatorType64&                       A64_;
   std::shared_ptr< Solver< OperatorType64 > > solver_;
   FunctionType64                              x64_, b64_;
};

// GeometricMultigridSolver (GeometricMultigridSolver.hpp:126-308)
// An open HIP graph capture of a context's stream (hg_graph_begin_capture).
// finish() ends it and returns the instantiated graph; leaving the scope
// without finish() (an exception inside the captured work) ends the capture and
// discards its graph, so the context's stream and the process-wide capture gate
// are released on every path.  No counterpart in the reference.
class CaptureScope
{
 public:
   explicit CaptureScope( hg_ctx* ctx )
   : ctx_( ctx )
   {
      check( ctx_, hg_graph_begin_capture( ctx_ ), "begin capture" );
   }
   CaptureScope( const CaptureScope& )            = delete;
   CaptureScope& operator=( const CaptureScope& ) = delete;
   hg_handle     finish()
   {
      hg_handle g = 0;
      open_       = false;
      check( ctx_, hg_graph_end_capture( ctx_, &g ), "end capture" );
      return g;
   }
   ~CaptureScope()
   {
      if ( !open_ )
         return;
      hg_handle g = 0;
      if ( hg_graph_end_capture( ctx_, &g ) == HG_OK && g )
         (void) hg_graph_destroy( ctx_, g );
   }

 private:
   hg_ctx* ctx_;
   bool    open_ = true;
};

template < class OperatorType >
class GeometricMultigridSolver : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;

   GeometricMultigridSolver( const std::shared_ptr< PrimitiveStorage >&                storage,
                             std::shared_ptr< Solver< OperatorType > >                smoother,
                             std::shared_ptr< Solver< OperatorType > >                coarseSolver,
                             std::shared_ptr< RestrictionOperator< FunctionType > >  restrictionOperator,
                             std::shared_ptr< ProlongationOperator< FunctionType > > prolongationOperator,
                             uint_t minLevel, uint_t maxLevel, uint_t preSmoothSteps = 3, uint_t postSmoothSteps = 3,
                             uint_t smoothIncrementOnCoarserGrids = 0, CycleType cycleType = CycleType::VCYCLE,
                             int nvec = 1 )
   : minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , pre_( preSmoothSteps )
   , post_( postSmoothSteps )
   , inc_( smoothIncrementOnCoarserGrids )
   , cycleType_( cycleType )
   , smoother_( std::move( smoother ) )
   , coarse_( std::move( coarseSolver ) )
   , restriction_( std::move( restrictionOperator ) )
   , prolongation_( std::move( prolongationOperator ) )
   , tmp_( "gmg_tmp", storage, minLevel, maxLevel, nvec )
   {}

   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      invokedLevel_ = level;
      hg_ctx* ctx   = x.ctx();
      region( ctx, "Geometric Multigrid Solver", true );
      solveRecursively( A, x, b, level );
      region( ctx, "Geometric Multigrid Solver", false );
   }

 private:
   // the timing regions of GeometricMultigridSolver.hpp:200-306 (recorded while
   // the context's timing tree is enabled)
   static void region( hg_ctx* ctx, const std::string& name, bool start )
   {
      check( ctx, start ? hg_timing_start( ctx, name.c_str() ) : hg_timing_stop( ctx, name.c_str() ), "timing" );
   }

   void solveRecursively( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level )
   {
      hg_ctx*           ctx = x.ctx();
      const std::string lv  = "Level " + std::to_string( level );
      if ( level == minLevel_ )
      {
         region( ctx, lv, true );
         region( ctx, "Coarse Grid Solver", true );
         coarse_->solve( A, x, b, minLevel_ );
         region( ctx, "Coarse Grid Solver", false );
         region( ctx, lv, false );
         return;
      }
      region( ctx, lv, true );
      const uint_t preSteps = pre_ + inc_ * ( invokedLevel_ - level );
      region( ctx, "Smoother", true );
      for ( uint_t i = 0; i < preSteps; ++i )
         smoother_->solve( A, x, b, level );
      region( ctx, "Smoother", false );
      A.apply( x, tmp_, level, flag_ );
      tmp_.assign( { 1.0, -1.0 }, { b, tmp_ }, level, flag_ );
      region( ctx, "Restriction", true );
      restriction_->restrict( tmp_, level, flag_ );
      region( ctx, "Restriction", false );
      b.assign( { 1.0 }, { tmp_ }, level - 1, flag_ );
      x.interpolate( 0, level - 1 );
      region( ctx, lv, false );
      solveRecursively( A, x, b, level - 1 );
      if ( cycleType_ == CycleType::WCYCLE )
         solveRecursively( A, x, b, level - 1 );
      region( ctx, lv, true );
      region( ctx, "Prolongation", true );
      prolongation_->prolongateAndAdd( x, level - 1, flag_ );
      region( ctx, "Prolongation", false );
      const uint_t postSteps = post_ + inc_ * ( invokedLevel_ - level );
      region( ctx, "Smoother", true );
      for ( uint_t i = 0; i < postSteps; ++i )
         smoother_->solve( A, x, b, level );
      region( ctx, "Smoother", false );
      region( ctx, lv, false );
   }

   uint_t                                                  minLevel_, maxLevel_, pre_, post_, inc_, invokedLevel_ = 0;
   CycleType                                               cycleType_;
   std::shared_ptr< Solver< OperatorType > >               smoother_, coarse_;
   std::shared_ptr< RestrictionOperator< FunctionType > >  restriction_;
   std::shared_ptr< ProlongationOperator< FunctionType > > prolongation_;
   FunctionType                                            tmp_;
   DoFType                                                 flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

// ---- P2-P1 Taylor-Hood Stokes --------------------------------------------------

// the pressure of a Taylor-Hood function has only Inner DoFs
// (P2P1TaylorHoodFunction.hpp:61, createAllInnerBC)
inline DoFType pressureFlag( DoFType flag )
{
   return ( flag & Inner ) ? All : DoFType( 0 );
}

namespace vertexdof {
// projectMean (p1functionspace/VertexDoFFunction.hpp:586-592): p -= sum(p) / #DoFs
inline void projectMean( const P1Function< double >& p, uint_t level )
{
   hg_handle s;
   int64_t   n   = 0;
   double    sum = 0.0;
   check( p.ctx(), hg_function_storage( p.ctx(), p.handle(), &s ), "projectMean" );
   check( p.ctx(), hg_p1_ndofs( p.ctx(), s, int( level ), &n ), "projectMean" );
   check( p.ctx(), hg_function_sum( p.ctx(), p.handle(), int( level ), All, &sum ), "projectMean" );
   check( p.ctx(), hg_function_add_const( p.ctx(), p.handle(), -sum / double( n ), int( level ), All ), "projectMean" );
}
} // namespace vertexdof

// P2VectorFunction<double>: the three components of a P2 vector field
template < typename VT >
class P2VectorFunction
{
 public:
   using valueType = typename ScalarOf< VT >::type; // the arithmetic type (float for f16 storage)
   using ValueType = valueType;

   P2VectorFunction( const std::string& name, const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel,
                     uint_t maxLevel, int nvec = 1 )
   {
      if ( nvec != 1 )
         throw std::invalid_argument( "P2 vector functions hold one vector" );
      for ( int k = 0; k < 3; ++k )
         c_[k] = std::make_unique< P2Function< VT > >( name + "_" + char( 'u' + k ), storage, minLevel, maxLevel );
   }
   // a view of three existing component handles (not owned)
   P2VectorFunction( hg_ctx* ctx, const hg_handle h[3] )
   {
      for ( int k = 0; k < 3; ++k )
         c_[k] = P2Function< VT >::borrow( ctx, h[k] );
   }
   const P2Function< VT >& operator[]( int k ) const { return *c_[k]; }
   hg_ctx*                 ctx() const { return c_[0]->ctx(); }

   void assign( const std::vector< ValueType >& scalars, const std::vector< std::reference_wrapper< const P2VectorFunction > >& fs,
                uint_t level, DoFType flag = All ) const
   {
      for ( int k = 0; k < 3; ++k )
         c_[k]->assign( scalars, component( fs, k ), level, flag );
   }
   void add( const std::vector< ValueType >& scalars, const std::vector< std::reference_wrapper< const P2VectorFunction > >& fs,
             uint_t level, DoFType flag = All ) const
   {
      for ( int k = 0; k < 3; ++k )
         c_[k]->add( scalars, component( fs, k ), level, flag );
   }
   void interpolate( ValueType constant, uint_t level, DoFType flag = All ) const
   {
      for ( int k = 0; k < 3; ++k )
         c_[k]->interpolate( constant, level, flag );
   }
   void setToZero( uint_t level ) const { interpolate( ValueType( 0 ), level, All ); }
   ValueType dotGlobal( const P2VectorFunction& o, uint_t level, DoFType flag = All ) const
   {
      ValueType s = 0;
      for ( int k = 0; k < 3; ++k )
         s += c_[k]->dotGlobal( *o.c_[k], level, flag );
      return s;
   }
   void multElementwise( const std::vector< std::reference_wrapper< const P2VectorFunction > >& fs, uint_t level,
                         DoFType flag = All ) const
   {
      for ( int k = 0; k < 3; ++k )
         c_[k]->multElementwise( component( fs, k ), level, flag );
   }
   // copyFrom<OtherT>: the values of another precision, cast
   template < typename OT >
   void copyFrom( const P2VectorFunction< OT >& o, uint_t level ) const
   {
      for ( int k = 0; k < 3; ++k )
         c_[k]->copyFrom( o[k], level );
   }

 private:
   static std::vector< std::reference_wrapper< const P2Function< VT > > >
       component( const std::vector< std::reference_wrapper< const P2VectorFunction > >& fs, int k )
   {
      std::vector< std::reference_wrapper< const P2Function< VT > > > out;
      for ( const auto& f : fs )
         out.push_back( f.get()[k] );
      return out;
   }
   std::unique_ptr< P2Function< VT > > c_[3];
};

// P2P1TaylorHoodFunction<double> (composites/P2P1TaylorHoodFunction.hpp): P2
// velocity uvw and P1 pressure p, whose DoFs are all Inner
template < typename VT >
class P2P1TaylorHoodFunction
{
 public:
   using valueType = VT;
   using ValueType = VT;

   P2P1TaylorHoodFunction( const std::string& name, const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel,
                           uint_t maxLevel, int nvec = 1 )
   : uvw_( std::make_unique< P2VectorFunction< VT > >( name + "_uvw", storage, minLevel, maxLevel, nvec ) )
   , p_( std::make_unique< P1Function< VT > >( name + "_p", storage, minLevel, maxLevel ) )
   {
      p_->setAllInner();
   }
   // a view of existing handles {u_x, u_y, u_z, p} (not owned)
   P2P1TaylorHoodFunction( hg_ctx* ctx, const hg_handle h[4] )
   : uvw_( std::make_unique< P2VectorFunction< VT > >( ctx, h ) )
   , p_( P1Function< VT >::borrow( ctx, h[3] ) )
   {
      p_->setAllInner();
   }
   const P2VectorFunction< VT >& uvw() const { return *uvw_; }
   const P1Function< VT >&       p() const { return *p_; }
   hg_ctx*                       ctx() const { return uvw_->ctx(); }

   void assign( const std::vector< VT >& scalars,
                const std::vector< std::reference_wrapper< const P2P1TaylorHoodFunction > >& fs, uint_t level,
                DoFType flag = All ) const
   {
      uvw_->assign( scalars, velocities( fs ), level, flag );
      if ( pressureFlag( flag ) )
         p_->assign( scalars, pressures( fs ), level, All );
   }
   void add( const std::vector< VT >& scalars, const std::vector< std::reference_wrapper< const P2P1TaylorHoodFunction > >& fs,
             uint_t level, DoFType flag = All ) const
   {
      uvw_->add( scalars, velocities( fs ), level, flag );
      if ( pressureFlag( flag ) )
         p_->add( scalars, pressures( fs ), level, All );
   }
   void interpolate( VT constant, uint_t level, DoFType flag = All ) const
   {
      uvw_->interpolate( constant, level, flag );
      if ( pressureFlag( flag ) )
         p_->interpolate( constant, level, All );
   }
   void setToZero( uint_t level ) const { interpolate( VT( 0 ), level, All ); }
   VT   dotGlobal( const P2P1TaylorHoodFunction& o, uint_t level, DoFType flag = All ) const
   {
      VT s = uvw_->dotGlobal( *o.uvw_, level, flag );
      if ( pressureFlag( flag ) )
         s += p_->dotGlobal( *o.p_, level, All );
      return s;
   }

 private:
   static std::vector< std::reference_wrapper< const P2VectorFunction< VT > > >
       velocities( const std::vector< std::reference_wrapper< const P2P1TaylorHoodFunction > >& fs )
   {
      std::vector< std::reference_wrapper< const P2VectorFunction< VT > > > out;
      for ( const auto& f : fs )
         out.push_back( f.get().uvw() );
      return out;
   }
   static std::vector< std::reference_wrapper< const P1Function< VT > > >
       pressures( const std::vector< std::reference_wrapper< const P2P1TaylorHoodFunction > >& fs )
   {
      std::vector< std::reference_wrapper< const P1Function< VT > > > out;
      for ( const auto& f : fs )
         out.push_back( f.get().p() );
      return out;
   }
   std::unique_ptr< P2VectorFunction< VT > > uvw_;
   std::unique_ptr< P1Function< VT > >       p_;
};

// P2ProjectNormalOperator (p2functionspace/P2ProjectNormalOperator.hpp:34-120,
// p1functionspace/freeslip/VertexDoFProjectNormal.hpp, edgedofspace/freeslip/
// EdgeDoFProjectNormal.hpp) with the radial normal of the spherical shell,
// n = x/|x| at the DoF's point (the shell map moves points along rays, so the
// computational and the physical point give the same n): u -= (u.n) n on every
// P2 DoF whose boundary type is in flag
class P2ProjectNormalOperator
{
 public:
   P2ProjectNormalOperator() = default;
   P2ProjectNormalOperator( const std::shared_ptr< PrimitiveStorage >&, uint_t, uint_t ) {}
   template < typename VT >
   void project( const P2VectorFunction< VT >& u, uint_t level, DoFType flag ) const
   {
      if ( !flag )
         return;
      const hg_handle h[3] = { u[0].handle(), u[1].handle(), u[2].handle() };
      check( u.ctx(), hg_p2_project_normal( u.ctx(), h, int( level ), flag ), "P2ProjectNormalOperator::project" );
   }
   void project( const P2P1TaylorHoodFunction< double >& f, uint_t level, DoFType flag ) const
   {
      project( f.uvw(), level, flag );
   }
   // the projection is symmetric: transpose or not, the same map
   void manipulate( const P2VectorFunction< double >& u, uint_t level, DoFType flag, bool /* transpose */ = false ) const
   {
      project( u, level, flag );
   }
};

namespace detail {
inline void stokesApply( hg_ctx* ctx, hg_handle op, const hg_handle src[4], const hg_handle dst[4], uint_t level,
                         DoFType flag, int mask, UpdateType update )
{
   check( ctx, hg_stokes_apply( ctx, op, src, dst, int( level ), flag, mask, update ), "Stokes apply" );
}
} // namespace detail

// P2ElementwiseBlendingFullViscousOperator (the velocity block
// 2 eta eps(u):eps(v) - 2/3 eta div u div v of a Stokes operator, whose device
// operator it shares; elementwiseoperators/P2ElementwiseBlendingFullViscousOperator.hpp)
class P2ElementwiseBlendingFullViscousOperator : public Operator< P2VectorFunction< double >, P2VectorFunction< double > >,
                                                 public OperatorWithInverseDiagonal< P2VectorFunction< double > >
{
 public:
   P2ElementwiseBlendingFullViscousOperator( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h,
                                             uint_t minLevel, uint_t maxLevel )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , h_( h )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   {}
   void apply( const P2VectorFunction< double >& src, const P2VectorFunction< double >& dst, uint_t level, DoFType flag,
               UpdateType updateType = Replace ) const override
   {
      const hg_handle s[4] = { src[0].handle(), src[1].handle(), src[2].handle(), 0 };
      const hg_handle d[4] = { dst[0].handle(), dst[1].handle(), dst[2].handle(), 0 };
      detail::stokesApply( ctx_, h_, s, d, level, flag, 1, updateType );
   }
   std::shared_ptr< P2VectorFunction< double > > getInverseDiagonalValues() const override
   {
      if ( !invDiag_ )
         const_cast< P2ElementwiseBlendingFullViscousOperator* >( this )->computeInverseDiagonalOperatorValues();
      return invDiag_;
   }
   void computeInverseDiagonalOperatorValues() override
   {
      invDiag_ = std::make_shared< P2VectorFunction< double > >( "inverseDiagonal", storage_, minLevel_, maxLevel_ );
      for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
      {
         const hg_handle d[3] = { ( *invDiag_ )[0].handle(), ( *invDiag_ )[1].handle(), ( *invDiag_ )[2].handle() };
         check( ctx_, hg_stokes_velocity_inverse_diagonal( ctx_, h_, int( L ), d ), "inverse diagonal" );
      }
   }

 private:
   std::shared_ptr< PrimitiveStorage >           storage_;
   hg_ctx*                                       ctx_;
   hg_handle                                     h_;
   uint_t                                        minLevel_, maxLevel_;
   std::shared_ptr< P2VectorFunction< double > > invDiag_;
};

// P2P1ElementwiseBlendingFullViscousStokesOperator
// (elementwiseoperators/P2P1ElementwiseBlendingStokesOperator.hpp:125-216) with
// viscosity eta(x) = exp(viscC0 + viscC1 |x|)
class P2P1ElementwiseBlendingFullViscousStokesOperator
: public Operator< P2P1TaylorHoodFunction< double >, P2P1TaylorHoodFunction< double > >
{
 public:
   using VelocityOperator_T = P2ElementwiseBlendingFullViscousOperator;

   P2P1ElementwiseBlendingFullViscousStokesOperator( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel,
                                                     uint_t maxLevel, double viscC0 = 0.0, double viscC1 = 0.0 )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( true )
   {
      check( ctx_, hg_stokes_create( ctx_, storage->handle(), int( minLevel ), int( maxLevel ), viscC0, viscC1, &h_ ),
             "P2P1ElementwiseBlendingFullViscousStokesOperator" );
      velocity_ = std::make_unique< VelocityOperator_T >( storage, h_, minLevel, maxLevel );
   }
   static std::unique_ptr< P2P1ElementwiseBlendingFullViscousStokesOperator >
       borrow( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h, uint_t minLevel, uint_t maxLevel )
   {
      return std::unique_ptr< P2P1ElementwiseBlendingFullViscousStokesOperator >(
          new P2P1ElementwiseBlendingFullViscousStokesOperator( storage, h, minLevel, maxLevel ) );
   }
   ~P2P1ElementwiseBlendingFullViscousStokesOperator() override
   {
      if ( owned_ && h_ )
         hg_operator_destroy( ctx_, h_ );
   }
   void apply( const P2P1TaylorHoodFunction< double >& src, const P2P1TaylorHoodFunction< double >& dst, uint_t level,
               DoFType flag, UpdateType updateType = Replace ) const override
   {
      const hg_handle s[4] = { src.uvw()[0].handle(), src.uvw()[1].handle(), src.uvw()[2].handle(), src.p().handle() };
      const hg_handle d[4] = { dst.uvw()[0].handle(), dst.uvw()[1].handle(), dst.uvw()[2].handle(), dst.p().handle() };
      detail::stokesApply( ctx_, h_, s, d, level, flag, 7, updateType );
   }
   const VelocityOperator_T& getA() const { return *velocity_; }
   // divT.apply(p, uvw): B^T p into the velocity
   void applyDivT( const P1Function< double >& p, const P2VectorFunction< double >& dst, uint_t level, DoFType flag,
                   UpdateType updateType = Replace ) const
   {
      const hg_handle s[4] = { 0, 0, 0, p.handle() };
      const hg_handle d[4] = { dst[0].handle(), dst[1].handle(), dst[2].handle(), 0 };
      detail::stokesApply( ctx_, h_, s, d, level, flag, 2, updateType );
   }
   // div.apply(uvw, p): B u into the pressure
   void applyDiv( const P2VectorFunction< double >& u, const P1Function< double >& dst, uint_t level, DoFType flag,
                  UpdateType updateType = Replace ) const
   {
      const hg_handle s[4] = { u[0].handle(), u[1].handle(), u[2].handle(), 0 };
      const hg_handle d[4] = { 0, 0, 0, dst.handle() };
      detail::stokesApply( ctx_, h_, s, d, level, flag, 4, updateType );
   }
   // values of P1PSPGInvDiagOperator (pspg_inv_diag_) and P1LumpedInvMassOperator
   const P1Function< double >& pspgInverseDiagonal() const { return pressureDiagonal( pspgInv_, 0 ); }
   const P1Function< double >& lumpedInverseMass() const { return pressureDiagonal( lumpedInv_, 1 ); }
   hg_handle                   handle() const { return h_; }
   const std::shared_ptr< PrimitiveStorage >& getStorage() const { return storage_; }

 private:
   P2P1ElementwiseBlendingFullViscousStokesOperator( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle h,
                                                     uint_t minLevel, uint_t maxLevel )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , h_( h )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , owned_( false )
   , velocity_( std::make_unique< VelocityOperator_T >( storage, h, minLevel, maxLevel ) )
   {}
   const P1Function< double >& pressureDiagonal( std::unique_ptr< P1Function< double > >& f, int kind ) const
   {
      if ( !f )
      {
         f = std::make_unique< P1Function< double > >( kind ? "lumpedInvMass" : "pspgInvDiag", storage_, minLevel_,
                                                       maxLevel_ );
         for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
            check( ctx_, hg_stokes_pressure_diagonal( ctx_, h_, int( L ), kind, f->handle() ), "pressure diagonal" );
      }
      return *f;
   }
   std::shared_ptr< PrimitiveStorage >                  storage_;
   hg_ctx*                                              ctx_ = nullptr;
   hg_handle                                            h_   = 0;
   uint_t                                               minLevel_, maxLevel_;
   bool                                                 owned_;
   std::unique_ptr< VelocityOperator_T >                velocity_;
   mutable std::unique_ptr< P1Function< double > >      pspgInv_, lumpedInv_;
};

// P2P1FullStokesFreeslipWrapperTemplate<P2ProjectNormalOperator, ...>
// (terraneo/operators/P2P1StokesOperatorWithWrapper.hpp:41-386) around the
// elementwise full-viscous Stokes operator, P the normal projection on the
// FreeslipBoundary DoFs:
//   getA()  = P A P   (velocity block; inverse diagonal of the unprojected A)
//   getBT() = P B^T,  getB() = B P,
//   apply   = the blocks on (P u, p), P applied to the velocity result and the
//             mean of the pressure result projected out.
// Results are written on flag only (the projection of a result touches the
// FreeslipBoundary DoFs that flag selects).
class P2P1FullStokesFreeslipWrapper : public Operator< P2P1TaylorHoodFunction< double >, P2P1TaylorHoodFunction< double > >
{
 public:
   using StokesOperator_T = P2P1ElementwiseBlendingFullViscousStokesOperator;

   class ViscousOperatorWrapped : public Operator< P2VectorFunction< double >, P2VectorFunction< double > >,
                                  public OperatorWithInverseDiagonal< P2VectorFunction< double > >
   {
    public:
      explicit ViscousOperatorWrapped( const P2P1FullStokesFreeslipWrapper& outer )
      : outer_( outer )
      {}
      void apply( const P2VectorFunction< double >& src, const P2VectorFunction< double >& dst, uint_t level, DoFType flag,
                  UpdateType updateType = Replace ) const override
      {
         outer_.applyA( src, dst, level, flag, updateType );
      }
      std::shared_ptr< P2VectorFunction< double > > getInverseDiagonalValues() const override
      {
         return outer_.stokes_->getA().getInverseDiagonalValues();
      }
      void computeInverseDiagonalOperatorValues() override
      {
         const_cast< StokesOperator_T::VelocityOperator_T& >( outer_.stokes_->getA() ).computeInverseDiagonalOperatorValues();
      }

    private:
      const P2P1FullStokesFreeslipWrapper& outer_;
   };
   using VelocityOperator_T = ViscousOperatorWrapped;

   P2P1FullStokesFreeslipWrapper( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel,
                                  std::shared_ptr< StokesOperator_T >        stokes,
                                  std::shared_ptr< P2ProjectNormalOperator > projection )
   : stokes_( std::move( stokes ) )
   , projection_( std::move( projection ) )
   , tmp_( std::make_unique< P2P1TaylorHoodFunction< double > >( "freeslip_tmp", storage, minLevel, maxLevel ) )
   , tmpdst_( std::make_unique< P2P1TaylorHoodFunction< double > >( "freeslip_tmpdst", storage, minLevel, maxLevel ) )
   , viscous_( *this )
   {}

   void apply( const P2P1TaylorHoodFunction< double >& src, const P2P1TaylorHoodFunction< double >& dst, uint_t level,
               DoFType flag, UpdateType updateType = Replace ) const override
   {
      projectedCopy( src.uvw(), level );
      tmp_->p().assign( { 1.0 }, { src.p() }, level, All );
      if ( updateType == Replace )
      {
         stokes_->apply( *tmp_, dst, level, flag, Replace );
         projection_->project( dst.uvw(), level, DoFType( flag & FreeslipBoundary ) );
      }
      else
      {
         stokes_->apply( *tmp_, *tmpdst_, level, flag, Replace );
         projection_->project( tmpdst_->uvw(), level, FreeslipBoundary );
         dst.add( { 1.0 }, { *tmpdst_ }, level, flag );
      }
      vertexdof::projectMean( dst.p(), level );
   }
   const VelocityOperator_T& getA() const { return viscous_; }
   // P B^T p into the velocity
   void applyDivT( const P1Function< double >& p, const P2VectorFunction< double >& dst, uint_t level, DoFType flag,
                   UpdateType updateType = Replace ) const
   {
      if ( updateType == Replace )
      {
         stokes_->applyDivT( p, dst, level, flag, Replace );
         projection_->project( dst, level, DoFType( flag & FreeslipBoundary ) );
         return;
      }
      stokes_->applyDivT( p, tmpdst_->uvw(), level, flag, Replace );
      projection_->project( tmpdst_->uvw(), level, FreeslipBoundary );
      dst.add( { 1.0 }, { tmpdst_->uvw() }, level, flag );
   }
   // B P u into the pressure
   void applyDiv( const P2VectorFunction< double >& u, const P1Function< double >& dst, uint_t level, DoFType flag,
                  UpdateType updateType = Replace ) const
   {
      projectedCopy( u, level );
      stokes_->applyDiv( tmp_->uvw(), dst, level, flag, updateType );
   }
   const P1Function< double >&                pspgInverseDiagonal() const { return stokes_->pspgInverseDiagonal(); }
   const P1Function< double >&                lumpedInverseMass() const { return stokes_->lumpedInverseMass(); }
   const StokesOperator_T&                    getStokesOperator() const { return *stokes_; }
   const std::shared_ptr< P2ProjectNormalOperator >& getProjection() const { return projection_; }

 private:
   // P A P u: the projected copy of u goes through the unprojected velocity block
   void applyA( const P2VectorFunction< double >& src, const P2VectorFunction< double >& dst, uint_t level, DoFType flag,
                UpdateType updateType ) const
   {
      projectedCopy( src, level );
      if ( updateType == Replace )
      {
         stokes_->getA().apply( tmp_->uvw(), dst, level, flag, Replace );
         projection_->project( dst, level, DoFType( flag & FreeslipBoundary ) );
         return;
      }
      stokes_->getA().apply( tmp_->uvw(), tmpdst_->uvw(), level, flag, Replace );
      projection_->project( tmpdst_->uvw(), level, FreeslipBoundary );
      dst.add( { 1.0 }, { tmpdst_->uvw() }, level, flag );
   }
   void projectedCopy( const P2VectorFunction< double >& u, uint_t level ) const
   {
      tmp_->uvw().assign( { 1.0 }, { u }, level, All );
      projection_->project( tmp_->uvw(), level, FreeslipBoundary );
   }

   std::shared_ptr< StokesOperator_T >                 stokes_;
   std::shared_ptr< P2ProjectNormalOperator >          projection_;
   std::unique_ptr< P2P1TaylorHoodFunction< double > > tmp_, tmpdst_;
   ViscousOperatorWrapped                              viscous_;
};

// FullStokesVelocityBlockBlockDiagonalPreconditioner
// (solvers/preconditioners/stokes/FullStokesVelocityBlockBlockDiagonalPreconditioner.hpp):
// the velocity solver applied to (A.getA(), x.uvw(), b.uvw())
template < class OperatorType >
class FullStokesVelocityBlockBlockDiagonalPreconditioner : public Solver< OperatorType >
{
 public:
   explicit FullStokesVelocityBlockBlockDiagonalPreconditioner(
       std::shared_ptr< Solver< typename OperatorType::VelocityOperator_T > > velocitySolver )
   : velocity_( std::move( velocitySolver ) )
   {}
   void solve( const OperatorType& A, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      velocity_->solve( A.getA(), x.uvw(), b.uvw(), level );
   }

 private:
   std::shared_ptr< Solver< typename OperatorType::VelocityOperator_T > > velocity_;
};

// UzawaSmoother, block variant without stabilisation (solvers/UzawaSmoother.hpp:330-470):
//   r_u = b_u - B^T p;  velocity smoothing of A u = r_u;  r_p = omega (b_p - B u);
//   p += D_pspg^-1 r_p  (with the mean of r_p and p projected out when asked)
template < class OperatorType >
class UzawaSmoother : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;

   UzawaSmoother( const std::shared_ptr< PrimitiveStorage >& storage, std::shared_ptr< Solver< OperatorType > > velocitySmoother,
                  uint_t minLevel, uint_t maxLevel, double relaxParam, DoFType flag = Inner | NeumannBoundary | FreeslipBoundary,
                  uint_t numVelocityIterations = 2, bool projectPressureMean = false )
   : velocity_( std::move( velocitySmoother ) )
   , relax_( relaxParam )
   , flag_( flag )
   , numVelocity_( numVelocityIterations )
   , project_( projectPressureMean )
   , r_( "uzawa_smoother_r", storage, minLevel, maxLevel )
   , tmp_( "uzawa_smoother_tmp", storage, minLevel, maxLevel )
   {}
   void setRelaxationParameter( double omega ) { relax_ = omega; }
   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      A.applyDivT( x.p(), r_.uvw(), level, flag_, Replace );
      r_.uvw().assign( { 1.0, -1.0 }, { b.uvw(), r_.uvw() }, level, flag_ );
      if ( projection_ )
         projection_->project( r_.uvw(), level, FreeslipBoundary );
      for ( uint_t i = 0; i < numVelocity_; ++i )
         velocity_->solve( A, x, r_, level );
      const DoFType pflag = pressureFlag( flag_ );
      if ( !pflag )
         return;
      A.applyDiv( x.uvw(), r_.p(), level, flag_, Replace );
      r_.p().assign( { relax_, -relax_ }, { b.p(), r_.p() }, level, pflag );
      if ( project_ )
         vertexdof::projectMean( r_.p(), level );
      tmp_.multElementwise( { A.pspgInverseDiagonal(), r_.p() }, level, pflag );
      x.p().add( { 1.0 }, { tmp_ }, level, pflag );
      if ( project_ )
         vertexdof::projectMean( x.p(), level );
   }

 protected:
   std::shared_ptr< P2ProjectNormalOperator > projection_;

 private:
   std::shared_ptr< Solver< OperatorType > > velocity_;
   double                                    relax_;
   DoFType                                   flag_;
   uint_t                                    numVelocity_;
   bool                                      project_;
   FunctionType                              r_;
   P1Function< double >                      tmp_;
};

// UzawaSmootherWithFreeSlipProjection (solvers/UzawaSmoother.hpp:480-613): the
// velocity residual r_u = b_u - B^T p is projected on the FreeslipBoundary DoFs
// before the velocity smoothing
template < class OperatorType >
class UzawaSmootherWithFreeSlipProjection : public UzawaSmoother< OperatorType >
{
 public:
   UzawaSmootherWithFreeSlipProjection( const std::shared_ptr< PrimitiveStorage >&  storage,
                                        std::shared_ptr< Solver< OperatorType > >   velocitySmoother,
                                        uint_t minLevel, uint_t maxLevel, double relaxParam,
                                        DoFType flag = Inner | NeumannBoundary | FreeslipBoundary,
                                        std::shared_ptr< P2ProjectNormalOperator > projection = nullptr,
                                        uint_t numVelocityIterations = 2, bool projectPressureMean = true )
   : UzawaSmoother< OperatorType >( storage, std::move( velocitySmoother ), minLevel, maxLevel, relaxParam, flag,
                                    numVelocityIterations, projectPressureMean )
   {
      this->projection_ = std::move( projection );
   }
};

// StokesPressureBlockPreconditioner<Op, P1LumpedInvMassOperator>
// (solvers/preconditioners/stokes/StokesPressureBlockPreconditioner.hpp): identity
// on the velocity, inverse lumped mass on the pressure
template < class OperatorType >
class StokesPressureBlockPreconditioner : public Solver< OperatorType >
{
 public:
   void solve( const OperatorType& A, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      x.assign( { 1.0 }, { b }, level, flag_ );
      x.p().multElementwise( { A.lumpedInverseMass(), b.p() }, level, pressureFlag( flag_ ) );
   }

 private:
   DoFType flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

// MinResSolver (solvers/MinresSolver.hpp:117-245)
template < class OperatorType >
class MinResSolver : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;

   MinResSolver( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel, uint_t maxIter,
                 double relativeTolerance, double absoluteTolerance,
                 std::shared_ptr< Solver< OperatorType > > preconditioner )
   : maxIter_( maxIter )
   , relTol_( relativeTolerance )
   , absTol_( absoluteTolerance )
   , prec_( std::move( preconditioner ) )
   {
      const char* names[10] = { "minres_vm", "minres_v",  "minres_vp", "minres_z",   "minres_zp",
                                "minres_wm", "minres_w",  "minres_wp", "minres_tmp", "minres_r" };
      for ( int i = 0; i < 10; ++i )
         f_[i] = std::make_unique< FunctionType >( names[i], storage, minLevel, maxLevel );
   }
   uint_t getIterations() const { return iterations_; }
   void   solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      auto &vm = f_[0], &v = f_[1], &vp = f_[2], &z = f_[3], &zp = f_[4], &wm = f_[5], &w = f_[6], &wp = f_[7],
           &r = f_[9];
      for ( auto& f : f_ )
         f->setToZero( level );
      A.apply( x, *r, level, flag_ );
      v->assign( { 1.0, -1.0 }, { b, *r }, level, flag_ );
      prec_->solve( A, *z, *v, level );
      double       gammaOld = 1.0;
      double       gammaNew = std::sqrt( z->dotGlobal( *v, level, flag_ ) );
      const double resStart = gammaNew;
      double       eta      = gammaNew;
      double       sOld = 0.0, sNew = 0.0, cOld = 1.0, cNew = 1.0;
      iterations_ = maxIter_;
      if ( gammaNew < absTol_ )
         return;
      for ( uint_t i = 0; i < maxIter_; ++i )
      {
         z->assign( { 1.0 / gammaNew }, { *z }, level, flag_ );
         A.apply( *z, *vp, level, flag_ );
         const double delta = vp->dotGlobal( *z, level, flag_ );
         vp->assign( { 1.0, -delta / gammaNew, -gammaNew / gammaOld }, { *vp, *v, *vm }, level, flag_ );
         zp->interpolate( 0, level, flag_ );
         prec_->solve( A, *zp, *vp, level );
         gammaOld           = gammaNew;
         gammaNew           = std::sqrt( zp->dotGlobal( *vp, level, flag_ ) );
         const double a0    = cNew * delta - cOld * sNew * gammaOld;
         const double a1    = std::sqrt( a0 * a0 + gammaNew * gammaNew );
         const double a2    = sNew * delta + cOld * cNew * gammaOld;
         const double a3    = sOld * gammaOld;
         cOld               = cNew;
         cNew               = a0 / a1;
         sOld               = sNew;
         sNew               = gammaNew / a1;
         wp->assign( { 1.0 / a1, -a3 / a1, -a2 / a1 }, { *z, *wm, *w }, level, flag_ );
         x.add( { cNew * eta }, { *wp }, level, flag_ );
         eta = -sNew * eta;
         // (vm, v, vp) <- (v, vp, vm); (wm, w, wp) <- (w, wp, wm); (z, zp) <- (zp, z)
         std::swap( vm, v );
         std::swap( v, vp );
         std::swap( wm, w );
         std::swap( w, wp );
         std::swap( z, zp );
         if ( std::abs( eta ) / resStart < relTol_ || std::abs( eta ) < absTol_ )
         {
            iterations_ = i;
            break;
         }
      }
   }

 private:
   uint_t                                    maxIter_, iterations_ = 0;
   double                                    relTol_, absTol_;
   std::shared_ptr< Solver< OperatorType > > prec_;
   std::unique_ptr< FunctionType >           f_[10];
   DoFType                                   flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

// P2P1StokesToP2P1StokesRestriction / Prolongation
// (gridtransferoperators/P2P1StokesToP2P1StokesRestriction.hpp, ...Prolongation.hpp):
// quadratic transfer of each velocity component, linear transfer of the pressure
class P2P1StokesToP2P1StokesRestriction : public RestrictionOperator< P2P1TaylorHoodFunction< double > >
{
 public:
   explicit P2P1StokesToP2P1StokesRestriction( bool projectMeanAfterRestriction = false )
   : project_( projectMeanAfterRestriction )
   {}
   void restrict( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      for ( int k = 0; k < 3; ++k )
         check( f.p().ctx(), hg_p2_restrict( f.p().ctx(), f.uvw()[k].handle(), int( sourceLevel ), flag ), "restrict" );
      if ( pressureFlag( flag ) )
         check( f.p().ctx(), hg_p1_restrict( f.p().ctx(), f.p().handle(), int( sourceLevel ), All ), "restrict" );
      if ( project_ )
         vertexdof::projectMean( f.p(), sourceLevel - 1 );
   }

 private:
   bool project_;
};
class P2P1StokesToP2P1StokesProlongation : public ProlongationOperator< P2P1TaylorHoodFunction< double > >
{
 public:
   explicit P2P1StokesToP2P1StokesProlongation( bool projectMeanAfterProlongation = false )
   : project_( projectMeanAfterProlongation )
   {}
   void prolongate( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      transfer( f, sourceLevel, flag, HG_REPLACE );
   }
   void prolongateAndAdd( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      transfer( f, sourceLevel, flag, HG_ADD );
   }

 private:
   void transfer( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag, int update ) const
   {
      hg_ctx* ctx = f.p().ctx();
      for ( int k = 0; k < 3; ++k )
         check( ctx, hg_p2_prolongate( ctx, f.uvw()[k].handle(), int( sourceLevel ), flag, update ), "prolongate" );
      if ( pressureFlag( flag ) )
         check( ctx, hg_p1_prolongate( ctx, f.p().handle(), int( sourceLevel ), All, update ), "prolongate" );
      if ( project_ )
         vertexdof::projectMean( f.p(), sourceLevel + 1 );
   }
   bool project_;
};

// P2P1StokesToP2P1StokesRestrictionWithFreeSlipProjection
// (P2P1StokesToP2P1StokesRestriction.hpp:110-129): restrict, then project the
// coarse velocity on the FreeslipBoundary DoFs and the coarse pressure mean out
class P2P1StokesToP2P1StokesRestrictionWithFreeSlipProjection : public P2P1StokesToP2P1StokesRestriction
{
 public:
   explicit P2P1StokesToP2P1StokesRestrictionWithFreeSlipProjection( std::shared_ptr< P2ProjectNormalOperator > projection )
   : P2P1StokesToP2P1StokesRestriction( false )
   , projection_( std::move( projection ) )
   {}
   void restrict( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      P2P1StokesToP2P1StokesRestriction::restrict( f, sourceLevel, flag );
      projection_->project( f, sourceLevel - 1, FreeslipBoundary );
      vertexdof::projectMean( f.p(), sourceLevel - 1 );
   }

 private:
   std::shared_ptr< P2ProjectNormalOperator > projection_;
};

// P2P1StokesToP2P1StokesProlongationWithFreeSlipProjection
// (P2P1StokesToP2P1StokesProlongation.hpp:145-178): prolongate, project the fine
// velocity and the fine pressure mean; prolongateAndAdd prolongates a copy of
// the coarse function in `temp` and adds it on flag
class P2P1StokesToP2P1StokesProlongationWithFreeSlipProjection : public P2P1StokesToP2P1StokesProlongation
{
 public:
   P2P1StokesToP2P1StokesProlongationWithFreeSlipProjection( std::shared_ptr< P2P1TaylorHoodFunction< double > > temp,
                                                             std::shared_ptr< P2ProjectNormalOperator >          projection )
   : P2P1StokesToP2P1StokesProlongation( false )
   , temp_( std::move( temp ) )
   , projection_( std::move( projection ) )
   {}
   void prolongate( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      P2P1StokesToP2P1StokesProlongation::prolongate( f, sourceLevel, flag );
      projection_->project( f, sourceLevel + 1, FreeslipBoundary );
      vertexdof::projectMean( f.p(), sourceLevel + 1 );
   }
   void prolongateAndAdd( const P2P1TaylorHoodFunction< double >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      temp_->assign( { 1.0 }, { f }, sourceLevel, All );
      prolongate( *temp_, sourceLevel, flag );
      f.assign( { 1.0, 1.0 }, { f, *temp_ }, sourceLevel + 1, flag );
   }

 private:
   std::shared_ptr< P2P1TaylorHoodFunction< double > > temp_;
   std::shared_ptr< P2ProjectNormalOperator >          projection_;
};

// P2toP2QuadraticVectorRestriction / Prolongation
// (gridtransferoperators/P2toP2QuadraticVectorRestriction.hpp, ...Prolongation.hpp):
// the quadratic transfers of each velocity component
// (VT: the value type of the transferred functions)
template < typename VT = double >
class P2toP2QuadraticVectorRestrictionT : public RestrictionOperator< P2VectorFunction< VT > >
{
 public:
   void restrict( const P2VectorFunction< VT >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      for ( int k = 0; k < 3; ++k )
         check( f.ctx(), hg_p2_restrict( f.ctx(), f[k].handle(), int( sourceLevel ), flag ), "restrict" );
   }
};
template < typename VT = double >
class P2toP2QuadraticVectorProlongationT : public ProlongationOperator< P2VectorFunction< VT > >
{
 public:
   void prolongate( const P2VectorFunction< VT >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      for ( int k = 0; k < 3; ++k )
         check( f.ctx(), hg_p2_prolongate( f.ctx(), f[k].handle(), int( sourceLevel ), flag, HG_REPLACE ), "prolongate" );
   }
   void prolongateAndAdd( const P2VectorFunction< VT >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      for ( int k = 0; k < 3; ++k )
         check( f.ctx(), hg_p2_prolongate( f.ctx(), f[k].handle(), int( sourceLevel ), flag, HG_ADD ), "prolongate" );
   }
};
using P2toP2QuadraticVectorRestriction  = P2toP2QuadraticVectorRestrictionT< double >;
using P2toP2QuadraticVectorProlongation = P2toP2QuadraticVectorProlongationT< double >;

// P2toP2QuadraticVector{Restriction,Prolongation}WithProjection with their default
// configuration (P2toP2QuadraticVectorRestriction.hpp:54-150,
// P2toP2QuadraticVectorProlongation.hpp:64-230: no pre-projection, post-projection
// allowed to change the destination): transfer, then project the result on the
// projectionFlag DoFs of the target level
template < typename VT = double >
class P2toP2QuadraticVectorRestrictionWithProjectionT : public P2toP2QuadraticVectorRestrictionT< VT >
{
 public:
   explicit P2toP2QuadraticVectorRestrictionWithProjectionT( std::shared_ptr< P2ProjectNormalOperator > projection,
                                                             DoFType projectionFlag = FreeslipBoundary )
   : projection_( std::move( projection ) )
   , projectionFlag_( projectionFlag )
   {}
   void restrict( const P2VectorFunction< VT >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      P2toP2QuadraticVectorRestrictionT< VT >::restrict( f, sourceLevel, flag );
      projection_->project( f, sourceLevel - 1, projectionFlag_ );
   }

 private:
   std::shared_ptr< P2ProjectNormalOperator > projection_;
   DoFType                                    projectionFlag_;
};
template < typename VT = double >
class P2toP2QuadraticVectorProlongationWithProjectionT : public P2toP2QuadraticVectorProlongationT< VT >
{
 public:
   explicit P2toP2QuadraticVectorProlongationWithProjectionT( std::shared_ptr< P2ProjectNormalOperator > projection,
                                                              DoFType projectionFlag = FreeslipBoundary )
   : projection_( std::move( projection ) )
   , projectionFlag_( projectionFlag )
   {}
   void prolongate( const P2VectorFunction< VT >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      P2toP2QuadraticVectorProlongationT< VT >::prolongate( f, sourceLevel, flag );
      projection_->project( f, sourceLevel + 1, projectionFlag_ );
   }
   void prolongateAndAdd( const P2VectorFunction< VT >& f, uint_t sourceLevel, DoFType flag ) const override
   {
      P2toP2QuadraticVectorProlongationT< VT >::prolongateAndAdd( f, sourceLevel, flag );
      projection_->project( f, sourceLevel + 1, projectionFlag_ );
   }

 private:
   std::shared_ptr< P2ProjectNormalOperator > projection_;
   DoFType                                    projectionFlag_;
};
using P2toP2QuadraticVectorRestrictionWithProjection  = P2toP2QuadraticVectorRestrictionWithProjectionT< double >;
using P2toP2QuadraticVectorProlongationWithProjection = P2toP2QuadraticVectorProlongationWithProjectionT< double >;

// The velocity block of the Stokes operator on FP32 or FP16 functions (FP32
// arithmetic; the reduced-precision half of a mixed-precision velocity
// solver), sharing the Stokes operator's device data.  With a projection it is
// the free-slip P A P of P2P1FullStokesFreeslipWrapper::getA().  The inverse
// diagonal is the FP64 one, cast.
template < typename VT >
class P2ElementwiseBlendingFullViscousOperatorT : public Operator< P2VectorFunction< VT >, P2VectorFunction< VT > >,
                                                  public OperatorWithInverseDiagonal< P2VectorFunction< VT > >
{
   using Scalar = typename ScalarOf< VT >::type;

 public:
   P2ElementwiseBlendingFullViscousOperatorT( const std::shared_ptr< PrimitiveStorage >& storage, hg_handle stokesOperator,
                                              uint_t minLevel, uint_t maxLevel,
                                              std::shared_ptr< P2ProjectNormalOperator > projection = nullptr )
   : storage_( storage )
   , ctx_( storage->ctx() )
   , h_( stokesOperator )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , projection_( std::move( projection ) )
   {
      if ( projection_ )
      {
         tmp_    = std::make_unique< P2VectorFunction< VT > >( "viscous_low_tmp", storage, minLevel, maxLevel );
         tmpdst_ = std::make_unique< P2VectorFunction< VT > >( "viscous_low_tmpdst", storage, minLevel, maxLevel );
      }
   }
   void apply( const P2VectorFunction< VT >& src, const P2VectorFunction< VT >& dst, uint_t level, DoFType flag,
               UpdateType updateType = Replace ) const override
   {
      if ( !projection_ )
      {
         raw( src, dst, level, flag, updateType );
         return;
      }
      tmp_->assign( { Scalar( 1 ) }, { src }, level, All );
      projection_->project( *tmp_, level, FreeslipBoundary );
      if ( updateType == Replace )
      {
         raw( *tmp_, dst, level, flag, Replace );
         projection_->project( dst, level, DoFType( flag & FreeslipBoundary ) );
         return;
      }
      raw( *tmp_, *tmpdst_, level, flag, Replace );
      projection_->project( *tmpdst_, level, FreeslipBoundary );
      dst.add( { Scalar( 1 ) }, { *tmpdst_ }, level, flag );
   }
   std::shared_ptr< P2VectorFunction< VT > > getInverseDiagonalValues() const override
   {
      if ( !invDiag_ )
         const_cast< P2ElementwiseBlendingFullViscousOperatorT* >( this )->computeInverseDiagonalOperatorValues();
      return invDiag_;
   }
   void computeInverseDiagonalOperatorValues() override
   {
      invDiag_ = std::make_shared< P2VectorFunction< VT > >( "inverseDiagonal_low", storage_, minLevel_, maxLevel_ );
      P2VectorFunction< double > d64( "inverseDiagonal64", storage_, minLevel_, maxLevel_ );
      for ( uint_t L = minLevel_; L <= maxLevel_; ++L )
      {
         const hg_handle d[3] = { d64[0].handle(), d64[1].handle(), d64[2].handle() };
         check( ctx_, hg_stokes_velocity_inverse_diagonal( ctx_, h_, int( L ), d ), "inverse diagonal" );
         invDiag_->copyFrom( d64, L );
      }
   }

 private:
   void raw( const P2VectorFunction< VT >& src, const P2VectorFunction< VT >& dst, uint_t level, DoFType flag,
             UpdateType updateType ) const
   {
      const hg_handle s[4] = { src[0].handle(), src[1].handle(), src[2].handle(), 0 };
      const hg_handle d[4] = { dst[0].handle(), dst[1].handle(), dst[2].handle(), 0 };
      detail::stokesApply( ctx_, h_, s, d, level, flag, 1, updateType );
   }
   std::shared_ptr< PrimitiveStorage >        storage_;
   hg_ctx*                                    ctx_;
   hg_handle                                  h_;
   uint_t                                     minLevel_, maxLevel_;
   std::shared_ptr< P2ProjectNormalOperator > projection_;
   std::unique_ptr< P2VectorFunction< VT > >  tmp_, tmpdst_;
   std::shared_ptr< P2VectorFunction< VT > >  invDiag_;
};

// A solver of a reduced-precision operator used on FP64 functions: b and the
// start vector are cast to the solver's type, the result is cast back (the
// precision boundary of a mixed-precision preconditioner inside an FP64 outer
// iteration, as the iterative-refinement driver of
// mixedPrecisionIterativeRefinement.cpp:163-172 casts around its inner GMG).
// With a projection the result is projected again in FP64: a projection applied
// in FP16 storage leaves normal components of the rounding's size, which the
// projected operator does not see and an outer iteration would accumulate.
template < class OperatorType64, class OperatorTypeLow >
class MixedPrecisionSolver : public Solver< OperatorType64 >
{
 public:
   using FunctionType64  = typename OperatorType64::srcType;
   using FunctionTypeLow = typename OperatorTypeLow::srcType;
   MixedPrecisionSolver( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel,
                         const OperatorTypeLow& Alow, std::shared_ptr< Solver< OperatorTypeLow > > inner,
                         std::shared_ptr< P2ProjectNormalOperator > projection = nullptr )
   : Alow_( Alow )
   , inner_( std::move( inner ) )
   , projection_( std::move( projection ) )
   , x_( "mixed_x", storage, minLevel, maxLevel )
   , b_( "mixed_b", storage, minLevel, maxLevel )
   {}
   void solve( const OperatorType64&, const FunctionType64& x, const FunctionType64& b, uint_t level ) override
   {
      b_.copyFrom( b, level );
      x_.copyFrom( x, level );
      inner_->solve( Alow_, x_, b_, level );
      x.copyFrom( x_, level );
      if constexpr ( std::is_same< FunctionType64, P2VectorFunction< double > >::value )
         if ( projection_ )
            projection_->project( x, level, FreeslipBoundary );
   }

 private:
   const OperatorTypeLow&                       Alow_;
   std::shared_ptr< Solver< OperatorTypeLow > > inner_;
   std::shared_ptr< P2ProjectNormalOperator >   projection_;
   FunctionTypeLow                              x_, b_;
};

// IdentityPreconditioner (solvers/preconditioners/IdentityPreconditioner.hpp): x = b
template < class OperatorType >
class IdentityPreconditioner : public Solver< OperatorType >
{
 public:
   void solve( const OperatorType&, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      x.assign( { 1.0 }, { b }, level, flag_ );
   }

 private:
   DoFType flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

// FunctionMultiplicationPreconditioner (solvers/FunctionMultiplicationPreconditioner.hpp):
// x = f * b elementwise with a fixed function f
template < class OperatorType >
class FunctionMultiplicationPreconditioner : public Solver< OperatorType >
{
 public:
   FunctionMultiplicationPreconditioner( std::shared_ptr< typename OperatorType::dstType > multFunction,
                                         DoFType flag = Inner | NeumannBoundary | FreeslipBoundary )
   : f_( std::move( multFunction ) )
   , flag_( flag )
   {}
   void solve( const OperatorType&, const typename OperatorType::srcType& x, const typename OperatorType::dstType& b,
               uint_t level ) override
   {
      x.multElementwise( { *f_, b }, level, flag_ );
   }

 private:
   std::shared_ptr< typename OperatorType::dstType > f_;
   DoFType                                           flag_;
};

// The Schur-complement operator of the free-slip Stokes wrapper (its
// SchurOperator_T, a P1 "K-mass" with k = 1/viscosity;
// terraneo/operators/P2P1StokesOperatorWithWrapper.hpp:233-288,388-395):
// (1/eta p, q) with eta the Stokes operator's viscosity at the blended points
// (4-point degree-2 rule), sharing the Stokes operator's device data.
class P1ElementwiseKMassOperator : public Operator< P1Function< double >, P1Function< double > >
{
 public:
   P1ElementwiseKMassOperator( hg_ctx* ctx, hg_handle stokesOperator )
   : ctx_( ctx )
   , h_( stokesOperator )
   {}
   void apply( const P1Function< double >& src, const P1Function< double >& dst, uint_t level, DoFType flag,
               UpdateType updateType = Replace ) const override
   {
      const hg_handle s[4] = { 0, 0, 0, src.handle() };
      const hg_handle d[4] = { 0, 0, 0, dst.handle() };
      detail::stokesApply( ctx_, h_, s, d, level, flag, 8, updateType );
   }
   // 1 / (M_k 1): the inverse lumped (row-sum) diagonal, for a
   // FunctionMultiplicationPreconditioner
   std::shared_ptr< P1Function< double > > inverseLumpedDiagonal( const std::shared_ptr< PrimitiveStorage >& storage,
                                                                  uint_t minLevel, uint_t maxLevel ) const
   {
      auto                 d = std::make_shared< P1Function< double > >( "kmass_lumped_inv", storage, minLevel, maxLevel );
      P1Function< double > one( "kmass_one", storage, minLevel, maxLevel );
      d->setAllInner();
      one.setAllInner();
      for ( uint_t L = minLevel; L <= maxLevel; ++L )
      {
         one.interpolate( 1.0, L, All );
         apply( one, *d, L, All, Replace );
         d->invertElementwise( L, All );
      }
      return d;
   }

 private:
   hg_ctx*   ctx_;
   hg_handle h_;
};

// BlockFactorisationPreconditioner (solvers/preconditioners/stokes/StokesBlockPreconditioners.hpp:366-448):
//   x.p = -S^-1 b.p;  x.uvw = A^-1 (b.uvw - B^T x.p)  (b.uvw projected when a projection is given)
// with S^-1 and A^-1 the given approximate solvers of the Schur operator and the velocity block
template < class OperatorType, class AOperatorType, class SchurOperatorType >
class BlockFactorisationPreconditioner : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;

   BlockFactorisationPreconditioner( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel,
                                     const SchurOperatorType&                              schurOp,
                                     std::shared_ptr< Solver< AOperatorType > >            ABlockSolver,
                                     std::shared_ptr< Solver< SchurOperatorType > >        schurSolver,
                                     uint_t                                                velocityIterations = 1,
                                     std::shared_ptr< P2ProjectNormalOperator >            projection         = nullptr,
                                     DoFType flag = Inner | NeumannBoundary | FreeslipBoundary )
   : schurOp_( schurOp )
   , A_( std::move( ABlockSolver ) )
   , S_( std::move( schurSolver ) )
   , velocityIterations_( velocityIterations )
   , projection_( std::move( projection ) )
   , flag_( flag )
   , tmp_( "BlockFactorisationPreconditioner_tmp", storage, minLevel, maxLevel )
   {}
   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      S_->solve( schurOp_, x.p(), b.p(), level );
      A.applyDivT( x.p(), tmp_.uvw(), level, flag_, Replace );
      tmp_.uvw().assign( { 1.0, 1.0 }, { b.uvw(), tmp_.uvw() }, level, flag_ );
      x.p().assign( { -1.0 }, { x.p() }, level, flag_ );
      if ( projection_ )
         projection_->project( tmp_.uvw(), level, FreeslipBoundary );
      for ( uint_t i = 0; i < velocityIterations_; ++i )
         A_->solve( A.getA(), x.uvw(), tmp_.uvw(), level );
   }

 private:
   const SchurOperatorType&                       schurOp_;
   std::shared_ptr< Solver< AOperatorType > >     A_;
   std::shared_ptr< Solver< SchurOperatorType > > S_;
   uint_t                                         velocityIterations_;
   std::shared_ptr< P2ProjectNormalOperator >     projection_;
   DoFType                                        flag_;
   FunctionType                                   tmp_;
};

// FGMRESSolver (solvers/FGMRESSolver.hpp:55-500): flexible GMRES, right
// preconditioned (the preconditioner may change between iterations), modified
// Gram-Schmidt Arnoldi, Givens rotations on the Hessenberg matrix; restarts
// every restartLength iterations; stops on the approximate residual (relative
// or absolute), on the Arnoldi breakdown tolerance, on the iteration hook, or
// after maxKrylowDim - 1 iterations.
template < class OperatorType >
class FGMRESSolver : public Solver< OperatorType >
{
 public:
   using FunctionType = typename OperatorType::srcType;
   using Hook         = std::function< bool( uint_t, double ) >; // (iteration, approximate residual) -> stop

   FGMRESSolver( const std::shared_ptr< PrimitiveStorage >& storage, uint_t minLevel, uint_t maxLevel,
                 uint_t maxKrylowDim = 1000, double approxRelativeTOL = 1e-16, double approxAbsoluteTOL = 1e-16,
                 std::shared_ptr< Solver< OperatorType > > preconditioner = nullptr, uint_t restartLength = 1000,
                 double arnoldiTOL = 1e-16 )
   : storage_( storage )
   , minLevel_( minLevel )
   , maxLevel_( maxLevel )
   , maxKrylowDim_( maxKrylowDim )
   , restartLength_( restartLength )
   , arnoldiTOL_( arnoldiTOL )
   , relTol_( approxRelativeTOL )
   , absTol_( approxAbsoluteTOL )
   , prec_( preconditioner ? std::move( preconditioner ) : std::make_shared< IdentityPreconditioner< OperatorType > >() )
   , r0_( "r0", storage, minLevel, maxLevel )
   {}
   void   setIterationHook( Hook hook ) { hook_ = std::move( hook ); }
   uint_t getIterations() const { return iterations_; }
   double getInitialResidual() const { return initRes_; }

   void solve( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level ) override
   {
      if ( level != vLevel_ )
      {
         V_.clear();
         vLevel_ = level;
      }
      r0_.setToZero( level );
      init( A, x, b, level, false );
      iterations_   = maxKrylowDim_ > 0 ? maxKrylowDim_ - 1 : 0; // iterations performed without an early stop
      double residual = absTol_ + 1.0;
      for ( uint_t j = 1; j < maxKrylowDim_; ++j )
      {
         if ( j % restartLength_ == 0 )
         {
            generateApproximation( x, level );
            init( A, x, b, level, true );
            continue;
         }
         const size_t k = j % restartLength_; // the Krylov index of this iteration
         // the preconditioner may work on coarser levels of z; the basis v lives on `level` alone
         while ( Z_.size() < k )
            Z_.push_back( std::make_unique< FunctionType >( "z", storage_, minLevel_, maxLevel_ ) );
         while ( V_.size() <= k )
            V_.push_back( std::make_unique< FunctionType >( "w", storage_, level, level ) );
         Z_[k - 1]->setToZero( level );
         prec_->solve( A, *Z_[k - 1], *V_[k - 1], level );
         A.apply( *Z_[k - 1], *V_[k], level, flag_ );
         // H is (k+1) x k, column major in rows of length k+1
         H_.resize( k );
         H_[k - 1].assign( k + 1, 0.0 );
         for ( size_t i = 0; i < k; ++i )
         {
            const double h = V_[k]->dotGlobal( *V_[i], level, flag_ );
            H_[k - 1][i]   = h;
            V_[k]->add( { -h }, { *V_[i] }, level, flag_ );
         }
         const double wNorm = std::sqrt( V_[k]->dotGlobal( *V_[k], level, flag_ ) );
         H_[k - 1][k]       = wNorm;
         residual           = hessenbergMinimizer();
         V_[k]->assign( { 1.0 / wNorm }, { *V_[k] }, level, flag_ );
         if ( hook_ && hook_( j, residual ) )
         {
            iterations_ = j;
            break;
         }
         if ( wNorm <= arnoldiTOL_ || residual <= absTol_ || residual / initRes_ <= relTol_ )
         {
            iterations_ = j;
            break;
         }
      }
      generateApproximation( x, level );
   }

 private:
   void init( const OperatorType& A, const FunctionType& x, const FunctionType& b, uint_t level, bool restart )
   {
      A.apply( x, r0_, level, flag_ );
      r0_.assign( { 1.0, -1.0 }, { b, r0_ }, level, flag_ );
      beta_ = std::sqrt( r0_.dotGlobal( r0_, level, flag_ ) );
      if ( !restart )
         initRes_ = beta_;
      H_.clear();
      rot_.clear();
      g_.assign( 1, beta_ );
      y_.clear();
      if ( V_.empty() )
         V_.push_back( std::make_unique< FunctionType >( "v0", storage_, level, level ) );
      V_[0]->assign( { 1.0 / beta_ }, { r0_ }, level, flag_ );
      if ( Z_.empty() )
         Z_.push_back( std::make_unique< FunctionType >( "z0", storage_, minLevel_, maxLevel_ ) );
   }
   // applies the stored rotations and a new one to the last column, returns
   // |residual| of the least-squares problem and sets y (back substitution)
   double hessenbergMinimizer()
   {
      const size_t k   = H_.size();
      auto&        col = H_[k - 1];
      for ( size_t i = 0; i + 1 < k; ++i )
      {
         const double c = rot_[i].first, s = rot_[i].second;
         const double a = col[i], b = col[i + 1];
         col[i]         = c * a + s * b;
         col[i + 1]     = -s * a + c * b;
      }
      double c = 1.0, s = 0.0;
      if ( col[k] != 0.0 )
      {
         const double r = std::sqrt( col[k - 1] * col[k - 1] + col[k] * col[k] );
         s              = col[k] / r;
         c              = col[k - 1] / r;
      }
      rot_.emplace_back( c, s );
      const double a = col[k - 1], b = col[k];
      col[k - 1]     = c * a + s * b;
      col[k]         = -s * a + c * b;
      g_.push_back( -s * g_[k - 1] );
      g_[k - 1] = c * g_[k - 1];
      y_.assign( k, 0.0 );
      for ( size_t i = k; i-- > 0; )
      {
         double t = g_[i];
         for ( size_t m = i + 1; m < k; ++m )
            t -= H_[m][i] * y_[m];
         y_[i] = t / H_[i][i];
      }
      return std::abs( g_[k] );
   }
   void generateApproximation( const FunctionType& x, uint_t level )
   {
      for ( size_t i = 0; i < y_.size(); ++i )
         x.add( { y_[i] }, { *Z_[i] }, level, flag_ );
      y_.clear();
   }

   std::shared_ptr< PrimitiveStorage >                 storage_;
   uint_t                                              minLevel_, maxLevel_, maxKrylowDim_, restartLength_;
   double                                              arnoldiTOL_, relTol_, absTol_;
   std::shared_ptr< Solver< OperatorType > >           prec_;
   FunctionType                                        r0_;
   std::vector< std::unique_ptr< FunctionType > >      V_, Z_;
   std::vector< std::vector< double > >                H_;
   std::vector< std::pair< double, double > >          rot_;
   std::vector< double >                               g_, y_;
   double                                              beta_ = 0.0, initRes_ = 0.0;
   uint_t                                              iterations_ = 0, vLevel_ = ~uint_t( 0 );
   Hook                                                hook_;
   DoFType                                             flag_ = Inner | NeumannBoundary | FreeslipBoundary;
};

} // namespace hyteg_amd
