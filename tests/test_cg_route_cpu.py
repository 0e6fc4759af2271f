"""CGSolver hands small P2 solves to one call of the C ABI (hg_p2_cg_assembled) only
where that call computes what its own loop would.  A C++ program built on the header
with the C ABI replaced by counting stubs, so no GPU is needed: every scenario prints
how often the one-launch solve, the operator's apply and the preconditioner ran."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <map>
#include "hyteg_amd/hyteg_amd.hpp"
using namespace hyteg_amd;

static int       nAssembled, nApply, nPrec, nDiag;
static hg_handle nextHandle = 100;
static std::map< hg_handle, std::pair< int, int > > levelsOf;
static std::map< hg_handle, hg_handle >             storages;
static hg_handle create( hg_handle storage, int lo, int hi )
{
   levelsOf[++nextHandle] = { lo, hi };
   storages[nextHandle]   = storage;
   return nextHandle;
}
static int level( hg_handle f, int l ) { return l >= levelsOf[f].first && l <= levelsOf[f].second ? HG_OK : HG_ERR_ARG; }
extern "C" {
const char* hg_last_error( const hg_ctx* ) { return "stub error"; }
int hg_slots_alloc( hg_ctx*, int, int* first ) { return *first = 0, HG_OK; }
int hg_slots_free( hg_ctx*, int, int ) { return HG_OK; }
int hg_slots_read( hg_ctx*, int, int n, double* out ) { return std::memset( out, 0, sizeof( double ) * n ), HG_OK; }
int hg_slots_cg_stop( hg_ctx*, int, int, double, double, int, int ) { return HG_OK; }
int hg_p2_function_create( hg_ctx*, hg_handle s, int lo, int hi, int, hg_handle* out ) { return *out = create( s, lo, hi ), HG_OK; }
int hg_function_destroy( hg_ctx*, hg_handle ) { return HG_OK; }
int hg_function_storage( hg_ctx*, hg_handle f, hg_handle* out ) { return *out = storages[f], HG_OK; }
int hg_function_nvec( hg_ctx*, hg_handle, int* n ) { return *n = 1, HG_OK; }
int hg_function_interpolate_const( hg_ctx*, hg_handle f, double, int l, int ) { return level( f, l ); }
int hg_function_assign( hg_ctx*, hg_handle f, int n, const double*, const hg_handle* g, int l, int )
{
   for ( int i = 0; i < n; ++i )
      if ( storages[g[i]] != storages[f] )
         return HG_ERR_ARG;
   return level( f, l );
}
int hg_function_dot_slot( hg_ctx*, hg_handle f, hg_handle, int l, int, int ) { return level( f, l ); }
int hg_function_mult( hg_ctx*, hg_handle f, hg_handle, hg_handle, int l, int ) { return ++nPrec, level( f, l ); }
int hg_function_lincomb_slots_gated( hg_ctx*, hg_handle f, int, const double*, const int*, const int*, const hg_handle*, int l,
                                     int, int, int )
{
   return level( f, l );
}
int hg_p2_apply( hg_ctx*, hg_handle, hg_handle, hg_handle, int, int, int ) { return ++nApply, HG_OK; }
int hg_p2_divkgrad_create( hg_ctx*, hg_handle, int, int, int, const double*, const double*, const double*, hg_handle* out )
{
   return *out = ++nextHandle, HG_OK;
}
int hg_operator_destroy( hg_ctx*, hg_handle ) { return HG_OK; }
int hg_p2_inverse_diagonal( hg_ctx*, hg_handle, int, hg_handle ) { return ++nDiag, HG_OK; }
int hg_p2_cg_assembled( hg_ctx*, hg_handle, hg_handle, hg_handle, int, int, int, double, double, int, int* its, int* applied )
{
   ++nAssembled;
   *its     = 3;
   *applied = 1;
   return HG_OK;
}
}

using Op  = P2ElementwiseBlendingDivKGradOperator;
using Fn  = P2Function< double >;
using Jac = InverseDiagonalPreconditioner< Op >;
struct ShiftedOp : Op
{
   using Op::Op;
   void apply( const Fn&, const Fn&, uint_t, DoFType, UpdateType = Replace ) const override { ++nApply; }
};
struct OtherPrec : Jac
{
   void solve( const Op&, const Fn&, const Fn&, uint_t ) override { ++nPrec; }
};

int main( int argc, char** argv )
{
   const std::string what = argv[1];
   hg_ctx*           ctx  = reinterpret_cast< hg_ctx* >( &nextHandle );
   auto              st = PrimitiveStorage::borrow( ctx, 1 ), other = PrimitiveStorage::borrow( ctx, 2 );
   Op                A( st, 0, 2 );
   ShiftedOp         B( st, 0, 2 );
   Fn                x( "x", st, 0, 2 ), b( "b", st, 0, 2 );
   std::shared_ptr< Solver< Op > > prec;
   if ( what == "jacobi" || what == "all_inner" )
      prec = std::make_shared< Jac >();
   if ( what == "preconditioner" )
      prec = std::make_shared< OtherPrec >();
   if ( what == "all_inner" )
      x.setAllInner();
   CGSolver< Op > cg( what == "storage" ? other : st, what == "level" ? 1 : 0, 2, 10, 1e-10, 1e-10, prec );
   if ( what == "fixed" )
      cg.setFixedIterations( true );
   int refused = 0;
   try
   {
      cg.solve( what == "operator" ? static_cast< const Op& >( B ) : A, x, b, 0 );
   } catch ( const std::exception& )
   {
      refused = 1;
   }
   std::printf( "%d %d %d %d %d\n", nAssembled, nApply > 0, nPrec > 0, refused, nDiag > 0 );
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("cg")
    src, exe = d / "cg.cpp", d / "cg"
    src.write_text(PROGRAM)
    # the stubs cover what the solver calls; the rest of the C ABI stays undefined
    subprocess.run(["g++", "-std=c++17", "-O0", "-no-pie", "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe),
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return str(exe)


def _run(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, check=True, timeout=60)
    return tuple(int(v) for v in r.stdout.split())


@pytest.mark.parametrize("what,expected", [
    # one-launch solves, apply ran, preconditioner ran, refused
    ("plain", (1, 0, 0, 0)),
    ("jacobi", (1, 0, 0, 0)),
    ("fixed", (0, 1, 0, 0)),
    # x with every DoF counted as Inner: the call's DoF types are the mesh's
    ("all_inner", (0, 1, 1, 0)),
    # classes derived from the operator and from the preconditioner override its steps
    ("operator", (0, 1, 0, 0)),
    ("preconditioner", (0, 1, 1, 0)),
    # a level or a storage that the solver was not made for
    ("level", (0, 0, 0, 1)),
    ("storage", (0, 1, 0, 1)),
])
def test_cg_uses_the_one_launch_solve_only_where_it_is_its_own(program, what, expected):
    assert _run(program, what)[:4] == expected


def test_a_one_launch_solve_leaves_the_inverse_diagonal_behind(program):
    """as the loop does: a later solve inside a graph capture cannot allocate it"""
    assert _run(program, "jacobi")[4] == 1
