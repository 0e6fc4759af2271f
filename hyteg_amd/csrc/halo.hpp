// Device-side geometry of owned macro-vertex/edge/face DoFs and their halo
// copies in the incident macro-cell lattices.  Replaces HyTeG's pack infos
// (VertexDoFPackInfo.hpp:192-700) by arithmetic on per-cell orientation data:
// an owned DoF is identified by its primitive and its local lattice
// coordinates; its position in an incident cell follows from which cell-local
// vertex each of the primitive's (sorted) vertices is.
#pragma once

#include "runtime.hpp"

namespace hg {

struct BndGeom
{
   const CellMeta* meta;
   const int32_t * fptr, *fcells, *eptr, *ecells, *vptr, *vcells;
   int64_t         mm, w, sc, fin, ein, eoff, foff;

   static BndGeom of( const Storage& st, const Lattice& l )
   {
      return BndGeom{ st.meta.p,
                      st.faceCellPtr.p,
                      st.faceCells.p,
                      st.edgeCellPtr.p,
                      st.edgeCells.p,
                      st.vertCellPtr.p,
                      st.vertCells.p,
                      l.mm,
                      l.w,
                      l.sc,
                      l.num.fin,
                      l.num.ein,
                      l.num.eoff,
                      l.num.foff };
   }
};

// (x, y) of index i in a triangle of width n (rows of n, n-1, ... points)
__device__ __forceinline__ void decodeTri( int64_t n, int64_t i, int64_t& x, int64_t& y )
{
   const double b  = 2.0 * double( n ) + 1.0;
   int64_t      yy = int64_t( floor( 0.5 * ( b - sqrt( b * b - 8.0 * double( i ) ) ) ) );
   if ( yy < 0 )
      yy = 0;
   while ( yy > 0 && triIndex( n, 0, yy ) > i )
      --yy;
   while ( triIndex( n, 0, yy + 1 ) <= i )
      ++yy;
   y = yy;
   x = i - triIndex( n, 0, yy );
}

// barycentric lattice weights t[0..3] in cell-local vertex order; (x,y,z) = t[1..3]
__device__ __forceinline__ void faceToCell( const CellMeta& m, int k, int64_t mm, int64_t fx, int64_t fy, int64_t t[4] )
{
   t[0] = t[1] = t[2] = t[3] = 0;
   t[m.fperm[k][0]] = mm - fx - fy;
   t[m.fperm[k][1]] = fx;
   t[m.fperm[k][2]] = fy;
}
__device__ __forceinline__ void edgeToCell( const CellMeta& m, int k, int64_t mm, int64_t s, int64_t t[4] )
{
   t[0] = t[1] = t[2] = t[3] = 0;
   t[m.eperm[k][0]] = mm - s;
   t[m.eperm[k][1]] = s;
}

// Calls f(c, x, y, z, cls) for every macro-cell incident to owned boundary DoF
// b (0 <= b < nb), in a fixed order; cls = local face k (0..3), 4 + local
// edge k, or 10 + local vertex k.
template < class F >
__device__ __forceinline__ void forEachIncident( const BndGeom& g, int64_t b, F&& f )
{
   int64_t t[4];
   if ( b < g.eoff )
   {
      for ( int32_t e = g.vptr[b]; e < g.vptr[b + 1]; ++e )
      {
         const int64_t c = g.vcells[2 * e];
         const int     k = g.vcells[2 * e + 1];
         t[0] = t[1] = t[2] = t[3] = 0;
         t[k]                      = g.mm;
         f( c, t[1], t[2], t[3], 10 + k );
      }
   }
   else if ( b < g.foff )
   {
      const int64_t eid = ( b - g.eoff ) / g.ein;
      const int64_t s   = ( b - g.eoff ) - eid * g.ein + 1;
      for ( int32_t e = g.eptr[eid]; e < g.eptr[eid + 1]; ++e )
      {
         const int64_t c = g.ecells[2 * e];
         const int     k = g.ecells[2 * e + 1];
         edgeToCell( g.meta[c], k, g.mm, s, t );
         f( c, t[1], t[2], t[3], 4 + k );
      }
   }
   else
   {
      const int64_t fid = ( b - g.foff ) / g.fin;
      const int64_t i   = ( b - g.foff ) - fid * g.fin;
      int64_t       a, bb;
      decodeTri( g.mm - 2, i, a, bb );
      for ( int32_t e = g.fptr[fid]; e < g.fptr[fid + 1]; ++e )
      {
         const int64_t c = g.fcells[2 * e];
         const int     k = g.fcells[2 * e + 1];
         faceToCell( g.meta[c], k, g.mm, a + 1, bb + 1, t );
         f( c, t[1], t[2], t[3], k );
      }
   }
}

// the same incidences by index: entries [e0, e1) of owned boundary DoF b, and
// the cell point (c; x, y, z) of entry e (the order of forEachIncident)
__device__ __forceinline__ void incidentRange( const BndGeom& g, int64_t b, int32_t& e0, int32_t& e1 )
{
   if ( b < g.eoff )
   {
      e0 = g.vptr[b];
      e1 = g.vptr[b + 1];
   }
   else if ( b < g.foff )
   {
      const int64_t eid = ( b - g.eoff ) / g.ein;
      e0                = g.eptr[eid];
      e1                = g.eptr[eid + 1];
   }
   else
   {
      const int64_t fid = ( b - g.foff ) / g.fin;
      e0                = g.fptr[fid];
      e1                = g.fptr[fid + 1];
   }
}
__device__ __forceinline__ int64_t incidentAt( const BndGeom& g, int64_t b, int32_t e, int64_t& x, int64_t& y,
                                               int64_t& z )
{
   int64_t t[4] = { 0, 0, 0, 0 };
   int64_t c;
   if ( b < g.eoff )
   {
      c    = g.vcells[2 * e];
      t[g.vcells[2 * e + 1]] = g.mm;
   }
   else if ( b < g.foff )
   {
      const int64_t eid = ( b - g.eoff ) / g.ein;
      const int64_t s   = ( b - g.eoff ) - eid * g.ein + 1;
      c                 = g.ecells[2 * e];
      edgeToCell( g.meta[c], g.ecells[2 * e + 1], g.mm, s, t );
   }
   else
   {
      const int64_t fid = ( b - g.foff ) / g.fin;
      const int64_t i   = ( b - g.foff ) - fid * g.fin;
      int64_t       a, bb;
      decodeTri( g.mm - 2, i, a, bb );
      c = g.fcells[2 * e];
      faceToCell( g.meta[c], g.fcells[2 * e + 1], g.mm, a + 1, bb + 1, t );
   }
   x = t[1];
   y = t[2];
   z = t[3];
   return c;
}

// class of a cell lattice point: -1 interior, 0..3 face, 4..9 edge, 10..13 vertex
__device__ __forceinline__ int pointClass( int64_t mm, int64_t x, int64_t y, int64_t z )
{
   const int64_t t[4] = { mm - x - y - z, x, y, z };
   int           nz = 0, zmask = 0;
   for ( int k = 0; k < 4; ++k )
      if ( t[k] == 0 )
      {
         ++nz;
         zmask |= 1 << k;
      }
   if ( nz == 0 )
      return -1;
   if ( nz == 1 )
   {
      // face k excludes vertex 3-k: faces (0,1,2), (0,1,3), (0,2,3), (1,2,3)
      for ( int k = 0; k < 4; ++k )
         if ( zmask == ( 1 << ( 3 - k ) ) )
            return k;
   }
   if ( nz == 2 )
   {
      // edges (0,1), (0,2), (1,2), (0,3), (1,3), (2,3): zero weights are the other two
      const int keep = ( ~zmask ) & 15;
      const int pairs[6] = { 3, 5, 6, 9, 10, 12 };
      for ( int k = 0; k < 6; ++k )
         if ( keep == pairs[k] )
            return 4 + k;
   }
   const int keep = ( ~zmask ) & 15;
   for ( int k = 0; k < 4; ++k )
      if ( keep == ( 1 << k ) )
         return 10 + k;
   return -1;
}

// ---- halo exchange ----------------------------------------------------------
// A halo copy's place in its cell follows from the primitive's orientation alone:
// the lattice keeps the cell-local offsets of the face and edge interiors for each
// orientation that the mesh has (haloOffsets), so an exchange costs one table load,
// one load and one store a value.  Bound by those loads' latency on small levels and
// by the scattered lines on large ones.  (Formed in the kernel -- 64-bit divisions,
// a square root for the row of a triangle, the tetrahedral index -- a pull took
// 14 us and a push 19 us at shell level 3, P2, and 1.21 and 0.65 ms at level 6.)
struct HaloGeom
{
   const CellMeta* meta;
   const int32_t * off, *faceInc, *edgePtr, *edgeInc, *vertPtr, *vertInc;
   int64_t         sc, base; // values of a cell lattice; first owned DoF
   uint32_t        fin, ein, nf, ne, nv, nfo; // points of a face / edge interior; counts; face orientations
   int64_t         eoff, foff;
   int32_t         vo[4]; // cell-local offsets of the vertices
   FastDiv         dfin, dein;
};

inline HaloGeom haloGeom( const Storage& st, const Lattice& l )
{
   const int64_t fin = l.num.fin, ein = l.num.ein, mm = l.mm;
   HaloGeom g;
   g.meta    = st.meta.p;
   g.off     = l.haloOffsets.p;
   g.faceInc = st.faceInc.p;
   g.edgePtr = st.edgeCellPtr.p;
   g.edgeInc = st.edgeInc.p;
   g.vertPtr = st.vertCellPtr.p;
   g.vertInc = st.vertCells.p;
   g.sc      = l.sc;
   g.base    = l.nc * l.sc;
   g.fin     = uint32_t( fin );
   g.ein     = uint32_t( ein );
   g.nf      = uint32_t( st.topo.nf );
   g.ne      = uint32_t( st.topo.ne );
   g.nv      = uint32_t( st.topo.nv );
   g.nfo     = uint32_t( st.faceOrient.size() );
   g.eoff    = l.num.eoff;
   g.foff    = l.num.foff;
   g.vo[0]   = 0;
   g.vo[1]   = int32_t( tetIndex( l.w, mm, 0, 0 ) );
   g.vo[2]   = int32_t( tetIndex( l.w, 0, mm, 0 ) );
   g.vo[3]   = int32_t( tetIndex( l.w, 0, 0, mm ) );
   g.dfin    = FastDiv( fin );
   g.dein    = FastDiv( ein );
   return g;
}

// whether a lattice's halo exchange runs on the offset tables: cell-local offsets in
// 32 bits and block counts within a grid (beyond that the general kernels run; the sums
// of a mesh with a face of three or more cells too, Storage::facesShared2)
inline bool haloTables( const Storage& st, const Lattice& l, int lv )
{
   const int64_t most = int64_t( 1 ) << 31, nf = st.topo.nf, ne = st.topo.ne, nv = st.topo.nv;
   // threads of a launch over n primitives of `per` values: whole workgroups each, or packed
   auto threads = []( int64_t per, int64_t n ) { return ( per / kBlock + 1 ) * kBlock * n; };
   return l.haloOffsets.p && threads( l.haloPerCell() << lv, l.nc ) / kBlock < most &&
          ( l.haloPerCell() << lv ) < most && threads( l.num.fin << lv, nf ) / kBlock < most &&
          ( ( l.haloPerCell() << lv ) >= kBlock / 2 || ( l.haloPerCell() << lv ) * l.nc < most ) &&
          ( ( l.num.fin << lv ) >= kBlock / 2 || ( l.num.fin << lv ) * nf < most ) && ( l.num.ein << lv ) * ne < most &&
          ( nv << lv ) < most;
}

// halo point p of cell c (4 fin face points, 6 ein edge points, 4 vertices): storage
// positions of its owner and of the copy
__device__ __forceinline__ void haloPoint( const HaloGeom& g, uint32_t c, uint32_t p, int64_t& src, int64_t& dst )
{
   const CellMeta& m = g.meta[c];
   int32_t         o;
   if ( p < 4 * g.fin )
   {
      const uint32_t k = uint32_t( p >= g.fin ) + uint32_t( p >= 2 * g.fin ) + uint32_t( p >= 3 * g.fin );
      p -= k * g.fin;
      o   = g.off[uint32_t( m.fcode[k] ) * g.fin + p];
      src = g.base + g.foff + int64_t( m.face[k] ) * g.fin + p;
   }
   else if ( ( p -= 4 * g.fin ) < 6 * g.ein )
   {
      uint32_t k = 0;
#pragma unroll
      for ( uint32_t i = 1; i < 6; ++i )
         k += uint32_t( p >= i * g.ein );
      p -= k * g.ein;
      o   = g.off[g.nfo * g.fin + uint32_t( m.ecode[k] ) * g.ein + p];
      src = g.base + g.eoff + int64_t( m.edge[k] ) * g.ein + p;
   }
   else
   {
      const uint32_t k = p - 6 * g.ein;
      o                = k == 0 ? g.vo[0] : ( k == 1 ? g.vo[1] : ( k == 2 ? g.vo[2] : g.vo[3] ) );
      src              = g.base + m.vert[k];
   }
   dst = c * g.sc + o;
}

} // namespace hg
